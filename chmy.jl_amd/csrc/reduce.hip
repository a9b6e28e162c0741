// Residual-norm reductions on the GPU: the reference's host-side
// maximum(abs.(interior(X))) (examples/stokes_3d_inc_ve_T.jl:172-175) and a
// deterministic f64 sum of squares.  max|x| is exact and order-independent:
// blocks reduce in registers (wave64 shuffles) and LDS, then combine with one
// 64-bit atomic max per block on the bit pattern (non-negative doubles order
// like their unsigned bits; NaN's bits exceed +inf's, so NaN propagates:
// fmax drops NaN, so a NaN seen anywhere is carried as a flag instead).
#include <mutex>

#include "common.hpp"

namespace chmy {

constexpr int kRB = 256;           // threads per reduction block
constexpr int kSumBlocks = 1024;   // fixed partial count: deterministic sum order

__device__ __forceinline__ double wave_max(double v) {
    for (int o = 32; o > 0; o >>= 1) v = fmax(v, __shfl_xor(v, o, 64));
    return v;
}
__device__ __forceinline__ double wave_sum(double v) {
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

struct MaxOut {
    unsigned long long* p[16];
};
__global__ void zero_u64(MaxOut o, int n) {
    if ((int)threadIdx.x < n) o.p[threadIdx.x][0] = 0ull;
}

// Work items of the sum of squares are (x-row, 256-element segment) pairs of
// the box; a wave takes kRW consecutive items at a time and issues all their
// loads (kRW x 4 per lane) before adding, so that each wave keeps 16 loads in
// flight.  Item bases are formed once per item; no per-element division is
// needed.
constexpr int kRowChunk = 4;   // 64-wide slices of an item
constexpr int kSeg = 64 * kRowChunk;
constexpr int kRW = 4;         // items of a wave in flight

// item -> (segment, row j, plane k) in 32-bit arithmetic (the host checks
// that the items of a box number below 2^32): 64-bit divisions per item
// cost more than the item's loads; one segment per row needs none for it.
__device__ __forceinline__ void item_rc(int64_t it, uint32_t nseg, uint32_t ny, int64_t& sg, int64_t& j,
                                        int64_t& k) {
    const uint32_t u = (uint32_t)it;
    const uint32_t r = nseg == 1 ? u : u / nseg;
    const uint32_t kk = r / ny;
    sg = (int64_t)(u - r * nseg);
    j = (int64_t)(r - kk * ny);
    k = (int64_t)kk;
}

// max|x| of up to kMaxMany fields in one launch (blockIdx.y = field).  A work
// item is a run of consecutive storage: as many whole rows of a plane as fit
// in 8 KB, padding included and masked, or an 8 KB segment of a longer row.
// A wave takes one item, reads it in 16 B granules at their own alignment
// (a run may start anywhere) with up to 9 loads a lane in flight, and only
// the granules at a run's two ends read element by element, so nothing
// outside the box's rows is touched beyond their padding.  Blocks combine
// with a 64-bit atomic max, taken only by a block whose maximum exceeds what
// the result already holds: all blocks' atomics go to one address, and there
// they take their turns.
// Bound by HBM on large fields and by the launch on small ones.  Measured, us
// (element-wise loads, one field a launch, every block's atomic -> now): four
// FP64 fields of 255^3 4 x 55 -> 149; four FP64 and six bf16 fields of
// 207x191x175 10 x 29 and ten clears -> 100 and one; three FP64 of 2047^2 3 x
// 25 -> 43; one of 250x230 14.4 (8 blocks) -> 6.5.  With up to 8 waves a SIMD
// the ten fields took 118.
constexpr int kMaxMany = 16;
constexpr int kRunBytes = 8192;
constexpr int kRunLoads = kRunBytes / (64 * 16) + 1;   // one more where the run starts inside a granule

struct MaxField {
    const char* p;        // first element of the box
    int64_t sy, sz;       // strides in elements
    int64_t nx, ny, nz;   // box
    int64_t rows;         // rows of a run, or 0: a run is a segment of one row
    int64_t runs, items;  // runs along a plane (bands of rows) or a row (segments); items in all
    int32_t dtype;
};
struct MaxArgs {
    MaxField f[kMaxMany];
    unsigned long long* out[kMaxMany];
};

// |x| as an unsigned integer: the bits without the sign order like the
// magnitudes, with NaN above infinity, so one integer max carries NaN too.
template <class U>
struct Granule {
    static constexpr int V = 16 / sizeof(U);
    U v[V];
};

template <class U>
__device__ __forceinline__ U max_item(const MaxField& f, int64_t item, U m) {
    using T = U;
    constexpr int V = Granule<U>::V;
    constexpr U mag = (U)~(U(1) << (8 * sizeof(U) - 1));
    const int lane = threadIdx.x & 63;
    const int64_t r = item / f.runs, u = item - r * f.runs;
    const T* base = reinterpret_cast<const T*>(f.p);
    int64_t len, pitch;   // elements of the run; x of element e is e % pitch, in the box when below nx
    if (f.rows) {         // r = plane, u = band of rows
        const int64_t j0 = u * f.rows, nr = f.ny - j0 < f.rows ? f.ny - j0 : f.rows;
        base += j0 * f.sy + r * f.sz;
        len = (nr - 1) * f.sy + f.nx;
        pitch = f.sy;
    } else {              // r = row of the box, u = segment
        const int64_t k = r / f.ny, j = r - k * f.ny, x0 = u * (kRunBytes / (int64_t)sizeof(T));
        base += x0 + j * f.sy + k * f.sz;
        len = f.nx - x0 < kRunBytes / (int64_t)sizeof(T) ? f.nx - x0 : kRunBytes / (int64_t)sizeof(T);
        pitch = len;
    }
    const int off = (int)((reinterpret_cast<uintptr_t>(base) & 15) / sizeof(T));   // elements into the first granule
    const uint32_t n = (uint32_t)len, w = (uint32_t)pitch, nx = (uint32_t)(f.rows ? f.nx : len);
    Granule<T> g[kRunLoads];
    // element e0 of the run is granule lane + 64 q's first (negative: before the run)
#pragma unroll
    for (int q = 0; q < kRunLoads; ++q) {
        const int e0 = V * (lane + 64 * q) - off;
        if (e0 >= 0 && e0 + V <= (int)n) {
            g[q] = *reinterpret_cast<const Granule<T>*>(__builtin_assume_aligned(base + e0, 16));
        } else {
#pragma unroll
            for (int v = 0; v < V; ++v) {
                const int e = e0 + v;
                g[q].v[v] = e >= 0 && e < (int)n ? base[e] : T{};
            }
        }
    }
#pragma unroll
    for (int q = 0; q < kRunLoads; ++q) {
        const int e0 = V * (lane + 64 * q) - off;
        uint32_t x = (uint32_t)(e0 < 0 ? 0 : e0);
        x = w < n ? x % w : x;
#pragma unroll
        for (int v = 0; v < V; ++v) {
            const U a = x < nx ? (U)(g[q].v[v] & mag) : U(0);   // zero outside the run
            m = a > m ? a : m;
            if (e0 + v >= 0) x = x + 1 == w ? 0 : x + 1;
        }
    }
    return m;
}

template <class U>
__device__ __forceinline__ U max_items(const MaxField& f) {
    U m = 0;
    for (int64_t it = (int64_t)blockIdx.x * (kRB / 64) + (threadIdx.x >> 6); it < f.items;
         it += (int64_t)gridDim.x * (kRB / 64))
        m = max_item<U>(f, it, m);
    return m;
}

__global__ void __launch_bounds__(kRB) maxabs_kernel(const MaxArgs a) {
    __shared__ double part[kRB / 64];
    const MaxField& f = a.f[blockIdx.y];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    double m;
    if (f.dtype == CHMY_F64) m = __longlong_as_double((long long)max_items<unsigned long long>(f));
    else if (f.dtype == CHMY_F32) m = (double)__uint_as_float(max_items<uint32_t>(f));
    else m = (double)bf16_to_f32(max_items<uint16_t>(f));
    const bool anynan = __any(m != m);
    m = wave_max(m);
    if (lane == 0) part[w] = anynan ? __longlong_as_double(0x7ff8000000000000ll) : m;
    __syncthreads();
    if (threadIdx.x == 0) {
        double v = part[0];
        bool nan = v != v;
        for (int q = 1; q < kRB / 64; ++q) {
            nan |= part[q] != part[q];
            v = fmax(v, part[q]);
        }
        if (nan) v = __longlong_as_double(0x7ff8000000000000ll);
        const unsigned long long bits = (unsigned long long)__double_as_longlong(v);
        unsigned long long* out = a.out[blockIdx.y];
        // a stale value only costs an atomic that changes nothing
        if (bits > __hip_atomic_load(out, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicMax(out, bits);
    }
}

// Sum of squares over (row, segment) items, in a fixed order: the
// grid is always kSumBlocks blocks, so which thread adds which element, and
// the order of every addition, depend on the box only.
template <class T>
__global__ void __launch_bounds__(kRB) sumsq_kernel(Box3 b, DF<T> f, double* partial) {
    __shared__ double part[kRB / 64];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int64_t nx = b.len[0], ny = b.len[1];
    const int64_t nseg = (nx + kSeg - 1) / kSeg;
    const int64_t items = ny * b.len[2] * nseg;
    const int64_t nw = (int64_t)gridDim.x * (kRB / 64);
    double s = 0.0;
    for (int64_t i0 = ((int64_t)blockIdx.x * (kRB / 64) + w) * kRW; i0 < items; i0 += nw * kRW) {
        const T* base[kRW];
        int64_t len[kRW];
#pragma unroll
        for (int u = 0; u < kRW; ++u) {
            const int64_t it = i0 + u;
            int64_t sg, j, k;
            item_rc(it, (uint32_t)nseg, (uint32_t)ny, sg, j, k);
            const bool ok = it < items;
            base[u] = ok ? &f(b.lo[0] + sg * kSeg, b.lo[1] + j, b.lo[2] + k) : nullptr;
            len[u] = ok ? (nx - sg * kSeg < kSeg ? nx - sg * kSeg : kSeg) : 0;
        }
        double a[kRW][kRowChunk];
#pragma unroll
        for (int u = 0; u < kRW; ++u)
#pragma unroll
            for (int q = 0; q < kRowChunk; ++q) {
                const int x = 64 * q + lane;
                a[u][q] = x < len[u] ? as_double(base[u][x]) : 0.0;
            }
#pragma unroll
        for (int u = 0; u < kRW; ++u)
#pragma unroll
            for (int q = 0; q < kRowChunk; ++q) s += a[u][q] * a[u][q];
    }
    s = wave_sum(s);
    if (lane == 0) part[w] = s;
    __syncthreads();
    if (threadIdx.x == 0) {
        double v = part[0];
        for (int q = 1; q < kRB / 64; ++q) v += part[q];
        partial[blockIdx.x] = v;
    }
}

__global__ void __launch_bounds__(kRB) sum_partials(const double* partial, int n, double* out) {
    __shared__ double part[kRB / 64];
    double s = 0.0;
    for (int q = threadIdx.x; q < n; q += kRB) s += partial[q];
    s = wave_sum(s);
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) {
        double v = part[0];
        for (int w = 1; w < kRB / 64; ++w) v += part[w];
        out[0] = v;
    }
}

// Library-held device scratch for reductions: one buffer per device, grown
// on demand, kept until process exit.
static std::mutex g_scratch_mu;
static void* g_scratch[64] = {nullptr};
static size_t g_scratch_sz[64] = {0};

static int scratch(size_t bytes, void** p) {
    int dev = 0;
    CHMY_HIP(hipGetDevice(&dev));
    if (dev < 0 || dev >= 64) return set_error(CHMY_E_ARG, "device index %d", dev);
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (g_scratch_sz[dev] < bytes) {
        if (g_scratch[dev]) CHMY_HIP(hipFree(g_scratch[dev]));
        g_scratch[dev] = nullptr;
        g_scratch_sz[dev] = 0;
        CHMY_HIP(hipMalloc(&g_scratch[dev], bytes));
        g_scratch_sz[dev] = bytes;
    }
    *p = g_scratch[dev];
    return 0;
}

static int reduce_box(const chmy_field_t* f, const chmy_box_t* box, Box3* out) {
    if (!f || !f->data) return set_error(CHMY_E_ARG, "field is NULL");
    if (f->nd < 1 || f->nd > 3) return set_error(CHMY_E_ARG, "field nd %d", f->nd);
    if (f->dtype != CHMY_F64 && f->dtype != CHMY_F32 && f->dtype != CHMY_BF16)
        return set_error(CHMY_E_DTYPE, "field dtype %d", f->dtype);
    chmy_box_t b;
    for (int d = 0; d < 3; ++d) { b.lo[d] = 1; b.len[d] = d < f->nd ? f->n[d] : 1; }
    if (box) b = *box;
    for (int d = 0; d < f->nd; ++d) {
        const int64_t H = f->halo[d];
        if (b.len[d] < 0 || b.lo[d] < 1 - 2 * H || b.lo[d] + b.len[d] - 1 > f->n[d] + 2 * H)
            return set_error(CHMY_E_BOX, "reduction box outside the storage of the field along dim %d", d);
    }
    *out = box3(b, f->nd);
    const int64_t items = out->len[1] * out->len[2] * ((out->len[0] + kSeg - 1) / kSeg);
    if (items >= (int64_t(1) << 32)) return set_error(CHMY_E_SIZE, "reduction box of 2^32 rows or more");
    return 0;
}

static MaxField max_field(const chmy_field_t& f, const Box3& b) {
    MaxField m;
    const int64_t es = f.dtype == CHMY_F64 ? 8 : f.dtype == CHMY_F32 ? 4 : 2;
    const DF<char> v = view<char>(f);   // strides in elements
    const int64_t o0 = v.p - static_cast<char*>(f.data);   // element offset of logical (0, 0, 0)
    m.p = static_cast<const char*>(f.data) + (o0 + b.lo[0] + b.lo[1] * v.sy + b.lo[2] * v.sz) * es;
    m.sy = v.sy;
    m.sz = v.sz;
    m.nx = b.len[0];
    m.ny = b.len[1];
    m.nz = b.len[2];
    m.dtype = f.dtype;
    const int64_t cap = kRunBytes / es;
    m.rows = f.nd >= 2 && v.sy <= cap ? cap / v.sy : 0;
    m.runs = m.rows ? (m.ny + m.rows - 1) / m.rows : (m.nx + cap - 1) / cap;
    m.items = no_work(b) ? 0 : m.runs * m.nz * (m.rows ? 1 : m.ny);
    if (m.runs < 1) m.runs = 1;
    return m;
}

static int max_launch(const MaxArgs& a, int n, hipStream_t s) {
    int64_t items = 0;
    MaxOut o;
    for (int q = 0; q < n; ++q) {
        items = items > a.f[q].items ? items : a.f[q].items;
        o.p[q] = a.out[q];
    }
    // a wave per item up to 4 waves a SIMD for each field, then rounds of them
    int64_t nb = (items + kRB / 64 - 1) / (kRB / 64), most = 4 * (int64_t)cu_count();
    nb = nb < 1 ? 1 : nb > most ? most : nb;
    hipLaunchKernelGGL(zero_u64, dim3(1), dim3(64), 0, s, o, n);
    hipLaunchKernelGGL(maxabs_kernel, dim3((unsigned)nb, (unsigned)n), dim3(kRB), 0, s, a);
    CHMY_HIP(hipGetLastError());
    return 0;
}

}  // namespace chmy

using namespace chmy;

extern "C" {

int chmy_maxabs_dev(const chmy_field_t* f, const chmy_box_t* box, double* out_dev, void* stream) {
    Box3 b;
    CHMY_TRY(reduce_box(f, box, &b));
    if (!out_dev) return set_error(CHMY_E_ARG, "out_dev is NULL");
    MaxArgs a;
    a.f[0] = max_field(*f, b);
    a.out[0] = reinterpret_cast<unsigned long long*>(out_dev);
    return max_launch(a, 1, (hipStream_t)stream);
}

int chmy_maxabs_many(int n, const chmy_field_t* f, double* out_dev, void* stream) {
    if (n < 0 || (n > 0 && (!f || !out_dev))) return set_error(CHMY_E_ARG, "chmy_maxabs_many: bad arguments");
    for (int q = 0; q < n; q += kMaxMany) {
        MaxArgs a;
        const int k = n - q < kMaxMany ? n - q : kMaxMany;
        for (int i = 0; i < k; ++i) {
            Box3 b;
            CHMY_TRY(reduce_box(&f[q + i], nullptr, &b));
            a.f[i] = max_field(f[q + i], b);
            a.out[i] = reinterpret_cast<unsigned long long*>(out_dev + q + i);
        }
        CHMY_TRY(max_launch(a, k, (hipStream_t)stream));
    }
    return 0;
}

int chmy_maxabs(const chmy_field_t* f, const chmy_box_t* box, double* out_host, void* stream) {
    if (!out_host) return set_error(CHMY_E_ARG, "out_host is NULL");
    void* p = nullptr;
    CHMY_TRY(scratch(kSumBlocks * sizeof(double) + 64, &p));
    double* d = static_cast<double*>(p) + kSumBlocks;
    CHMY_TRY(chmy_maxabs_dev(f, box, d, stream));
    CHMY_HIP(hipMemcpyAsync(out_host, d, sizeof(double), hipMemcpyDeviceToHost, (hipStream_t)stream));
    CHMY_HIP(hipStreamSynchronize((hipStream_t)stream));
    return 0;
}

int chmy_sumsq(const chmy_field_t* f, const chmy_box_t* box, double* out_host, void* stream) {
    Box3 b;
    CHMY_TRY(reduce_box(f, box, &b));
    if (!out_host) return set_error(CHMY_E_ARG, "out_host is NULL");
    void* p = nullptr;
    CHMY_TRY(scratch(kSumBlocks * sizeof(double) + 64, &p));
    double* partial = static_cast<double*>(p);
    double* res = partial + kSumBlocks;
    hipStream_t s = (hipStream_t)stream;
    if (f->dtype == CHMY_BF16)
        hipLaunchKernelGGL(sumsq_kernel<bf16s>, dim3(kSumBlocks), dim3(kRB), 0, s, b, view<bf16s>(*f), partial);
    else if (f->dtype == CHMY_F64)
        hipLaunchKernelGGL(sumsq_kernel<double>, dim3(kSumBlocks), dim3(kRB), 0, s, b, view<double>(*f), partial);
    else
        hipLaunchKernelGGL(sumsq_kernel<float>, dim3(kSumBlocks), dim3(kRB), 0, s, b, view<float>(*f), partial);
    hipLaunchKernelGGL(sum_partials, dim3(1), dim3(kRB), 0, s, partial, kSumBlocks, res);
    CHMY_HIP(hipGetLastError());
    CHMY_HIP(hipMemcpyAsync(out_host, res, sizeof(double), hipMemcpyDeviceToHost, s));
    CHMY_HIP(hipStreamSynchronize(s));
    return 0;
}

}  // extern "C"
