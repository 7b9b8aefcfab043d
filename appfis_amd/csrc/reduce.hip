// Box reductions (SUM / MIN / MAX) in a single pass.
//
// Replaces Execute{1,2,3}DReduceGPU + Kernel*DReduce* + KernelReduce*Loop of the
// reference (Appfis/Runtime_CUDA.hpp:554-740, 1249-1666), whose first pass scans the
// whole padded array with %,/ index math, then loops log_256 passes and copies one
// scalar back.  Here: waves stride over the Config box's rows only, per-thread accumulation
// in a wide type, a wave64 DPP reduction, one LDS stage per block, per-block
// partials, and the last block to arrive (atomic ticket) combines the partials in a
// fixed order -- so the result is deterministic and never leaves the device unless
// the host asked for it.
//
// Semantics kept from the reference CPU path (Appfis/Runtime.hpp:598-913): MAX
// starts at numeric_limits<T>::min(), MIN at numeric_limits<T>::max().  SUM is
// widened (int64 for integer types, compensated FP64 for floats) instead of being
// accumulated in T; the T-typed result is the widened sum rounded once.
#include "common.hpp"

#include <algorithm>
#include <cfloat>
#include <climits>
#include <mutex>

using namespace appfis;

namespace {

constexpr int MAX_RB = 1024;  // threads per block, at most
constexpr int MAX_BLOCKS = 2048;
constexpr int U = 4;  // steps of a wave in flight

struct Box {
    int d0, d1;             // padded extents along x, y
    int s0, s1, s2;         // box start
    int n0, n1, n2;         // box extents
};

// How the waves of a launch share the box.  A row of the box (n0 contiguous elements) is cut
// into chunks of V elements; a wave takes `lanes` consecutive chunks of 64 / lanes
// consecutive rows at a time, `segs` such steps to a row (lanes = 64 unless the row is short).
struct Split {
    uint64_t rows, items;  // rows of the box; steps of a wave over the whole box
    int chunks;            // per row
    int log_lanes, segs;
};

// V consecutive elements, at any address that is aligned for one of them
template <typename T, int V> struct Chunk;
template <typename T> struct Chunk<T, 1> {
    T v[1];
    __device__ void load(const T* p) { v[0] = *p; }
};
typedef unsigned int u32x4_any __attribute__((ext_vector_type(4), aligned(1), may_alias));
template <typename T, int V> struct Chunk {
    static_assert(V * sizeof(T) == 16, "one 16-byte load");
    T v[V];
    __device__ void load(const T* p)
    {
        const u32x4_any w = *reinterpret_cast<const u32x4_any*>(p);
        __builtin_memcpy(v, &w, 16);
    }
};

// --- compensated FP64 pair (Neumaier / TwoSum) ---------------------------------------
struct KSum {
    double s, c;
};
__device__ inline void two_sum_add(KSum& a, double x)
{
    double t = __dadd_rn(a.s, x);
    double bp = __dsub_rn(t, a.s);
    double err = __dadd_rn(__dsub_rn(a.s, __dsub_rn(t, bp)), __dsub_rn(x, bp));
    a.s = t;
    a.c = __dadd_rn(a.c, err);
}
__device__ inline KSum ksum_merge(KSum a, KSum b)
{
    two_sum_add(a, b.s);
    a.c = __dadd_rn(a.c, b.c);
    return a;
}

// wave reductions (DPP tree of common.hpp; the total is in lane WAVE_TOTAL_LANE)
template <typename T>
__device__ inline T wave_max(T v, T identity)
{
    return wave_reduce(v, identity, [](T a, T b) { return b > a ? b : a; });
}
template <typename T>
__device__ inline T wave_min(T v, T identity)
{
    return wave_reduce(v, identity, [](T a, T b) { return b < a ? b : a; });
}
__device__ inline long long wave_sum_i64(long long v)
{
    return wave_reduce(v, 0LL, [](long long a, long long b) { return a + b; });
}
__device__ inline KSum wave_sum_k(KSum v)
{
    return wave_reduce(v, KSum{0.0, 0.0}, [](KSum a, KSum b) { return ksum_merge(a, b); });
}

template <typename T> struct Lim;
template <> struct Lim<uint8_t> { static constexpr uint8_t lo = 0, hi = UCHAR_MAX; };
template <> struct Lim<int32_t> { static constexpr int32_t lo = INT_MIN, hi = INT_MAX; };
template <> struct Lim<float> { static constexpr float lo = FLT_MIN, hi = FLT_MAX; };
template <> struct Lim<double> { static constexpr double lo = DBL_MIN, hi = DBL_MAX; };

template <typename T, int OP> struct Ops;
// MAX/MIN of uint8 carry an int accumulator so every partial is a 4- or 8-byte word.
template <typename T> struct Wide { using type = T; };
template <> struct Wide<uint8_t> { using type = int; };

template <typename T> struct Ops<T, APPFIS_MAX> {
    using A = typename Wide<T>::type;
    __device__ static A init() { return Lim<T>::lo; }
    __device__ static void add(A& a, T v) { a = (A)v > a ? (A)v : a; }
    __device__ static A merge(A a, A b) { return b > a ? b : a; }
    __device__ static A wave(A a) { return wave_max(a, init()); }
};
template <typename T> struct Ops<T, APPFIS_MIN> {
    using A = typename Wide<T>::type;
    __device__ static A init() { return Lim<T>::hi; }
    __device__ static void add(A& a, T v) { a = (A)v < a ? (A)v : a; }
    __device__ static A merge(A a, A b) { return b < a ? b : a; }
    __device__ static A wave(A a) { return wave_min(a, init()); }
};
template <typename T> struct OpsSumInt {
    using A = long long;
    __device__ static A init() { return 0; }
    __device__ static void add(A& a, T v) { a += (long long)v; }
    __device__ static A merge(A a, A b) { return a + b; }
    __device__ static A wave(A a) { return wave_sum_i64(a); }
};
template <typename T> struct OpsSumFp {
    using A = KSum;
    __device__ static A init() { return KSum{0.0, 0.0}; }
    __device__ static void add(A& a, T v) { two_sum_add(a, (double)v); }
    __device__ static A merge(A a, A b) { return ksum_merge(a, b); }
    __device__ static A wave(A a) { return wave_sum_k(a); }
};
template <> struct Ops<uint8_t, APPFIS_SUM> : OpsSumInt<uint8_t> {};
template <> struct Ops<int32_t, APPFIS_SUM> : OpsSumInt<int32_t> {};
template <> struct Ops<float, APPFIS_SUM> : OpsSumFp<float> {};
template <> struct Ops<double, APPFIS_SUM> : OpsSumFp<double> {};

// Output conversion: MAX/MIN write T; SUM writes the wide result (int64 or double).
template <typename A> __device__ inline void write_wide(void* out, A a);
template <> __device__ inline void write_wide<long long>(void* out, long long a) { *(long long*)out = a; }
template <> __device__ inline void write_wide<KSum>(void* out, KSum a) { *(double*)out = __dadd_rn(a.s, a.c); }

template <typename T, int OP> __device__ inline void write_result(void* out, typename Ops<T, OP>::A a)
{
    if constexpr (OP == APPFIS_SUM) write_wide(out, a);
    else *(T*)out = (T)a;
}

// Partials written by other blocks are read past the (non-coherent) L1.
template <typename A> __device__ inline A load_l2(const A* p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <> __device__ inline KSum load_l2<KSum>(const KSum* p)
{
    KSum k;
    k.s = __hip_atomic_load(&p->s, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    k.c = __hip_atomic_load(&p->c, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return k;
}

// One chunk of a row: its elements from `skip` on (the last chunk of a row ends with the row
// and overlaps the one before it, whose elements it skips).
template <typename T, int OP, int V>
__device__ __forceinline__ void add_chunk(typename Ops<T, OP>::A& acc, const Chunk<T, V>& c, int skip)
{
    using O = Ops<T, OP>;
    if constexpr (sizeof(T) == 1 && OP == APPFIS_SUM && V == 16) {
        // sums of four bytes at a time; at most 16 * 255
        uint32_t w[4], sum = 0;
        __builtin_memcpy(w, c.v, 16);
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const int low = skip - 4 * q;  // bytes of this word to leave out
            const uint32_t keep = low <= 0 ? ~0u : low >= 4 ? 0u : ~0u << (8 * low);
            sum = __builtin_amdgcn_sad_u8(w[q] & keep, 0u, sum);
        }
        acc += (long long)sum;
    } else {
#pragma unroll
        for (int e = 0; e < V; e++)
            if (V == 1 || e >= skip) O::add(acc, c.v[e]);
    }
}

// The pass over the box reads each row in 16-byte loads (V = 16 / sizeof(T); V = 1 for rows
// shorter than one), consecutive lanes consecutive chunks, U steps of a wave in flight, and
// finds a row's address once per step instead of dividing for every element: 8192 x 8192
// bytes take 22 us against 163 (3.0 TB/s), 1024 x 1024 doubles 11 against 23, 512^3
// floats 150 against 402.
template <typename T, int OP, int V>
__global__ __launch_bounds__(MAX_RB) void k_reduce(const T* __restrict__ data, Box b, Split sp,
                                               typename Ops<T, OP>::A* partials, unsigned* ticket, void* out)
{
    using O = Ops<T, OP>;
    using A = typename O::A;
    __shared__ A lds[MAX_RB / 64];
    __shared__ bool is_last;
    A acc = O::init();
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    const int bwaves = (int)blockDim.x / 64;
    const uint64_t nwaves = (uint64_t)gridDim.x * bwaves;
    const uint64_t wave = (uint64_t)blockIdx.x * bwaves + (unsigned)__builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int sub = lane >> sp.log_lanes, in = lane & ((1 << sp.log_lanes) - 1);
    for (uint64_t t = wave; t < sp.items; t += U * nwaves) {
        Chunk<T, V> c[U];
        int skip[U];
#pragma unroll
        for (int u = 0; u < U; u++) {
            const uint64_t item = t + u * nwaves;
            uint64_t group = item, seg = 0;
            if (sp.segs > 1) {
                group = item < (1ULL << 32) ? (uint64_t)((uint32_t)item / (uint32_t)sp.segs) : item / (uint64_t)sp.segs;
                seg = item - group * (uint64_t)sp.segs;
            }
            const uint64_t row = (group << (6 - sp.log_lanes)) + sub;
            const int ch = (int)((seg << sp.log_lanes) + in);
            skip[u] = V;
            if (item < sp.items && row < sp.rows && ch < sp.chunks) {
                const uint64_t k = b.n2 == 1 ? 0
                                   : row < (1ULL << 32) ? (uint64_t)((uint32_t)row / (uint32_t)b.n1)
                                                        : row / (uint64_t)b.n1;
                const uint64_t j = row - k * (uint64_t)b.n1;
                const int first = ch * V, at = first <= b.n0 - V ? first : b.n0 - V;
                skip[u] = first - at;
                c[u].load(data + (size_t)(at + b.s0) +
                          (size_t)b.d0 * ((size_t)(j + b.s1) + (size_t)b.d1 * (size_t)(k + b.s2)));
            }
        }
#pragma unroll
        for (int u = 0; u < U; u++)
            if (skip[u] < V) add_chunk<T, OP, V>(acc, c[u], skip[u]);
    }
    acc = O::wave(acc);
    if (lane == WAVE_TOTAL_LANE) lds[wid] = acc;
    __syncthreads();
    if (threadIdx.x == 0) {
        A blk = lds[0];
        for (int w = 1; w < bwaves; w++) blk = O::merge(blk, lds[w]);
        if (gridDim.x == 1) {
            write_result<T, OP>(out, blk);
            return;
        }
        partials[blockIdx.x] = blk;
        __threadfence();
        unsigned prev = atomicAdd(ticket, 1u);
        is_last = (prev == gridDim.x - 1);
    }
    if (gridDim.x == 1) return;
    __syncthreads();
    if (!is_last) return;
    __threadfence();
    // last block: combine partials in a fixed order (thread t takes t, t + blockDim.x, ...)
    A v = O::init();
    for (unsigned p = threadIdx.x; p < gridDim.x; p += blockDim.x) {
        v = O::merge(v, load_l2(partials + p));
    }
    v = O::wave(v);
    if (lane == WAVE_TOTAL_LANE) lds[wid] = v;
    __syncthreads();
    if (threadIdx.x == 0) {
        A r = lds[0];
        for (int w = 1; w < bwaves; w++) r = O::merge(r, lds[w]);
        write_result<T, OP>(out, r);
        *ticket = 0u;  // ready for the next reduction on this context
    }
}

// Layout of a reduction's scratch: [0,256) ticket, [256, 256 + MAX_BLOCKS*16) partials
// (one 16-byte slot per block at most: KSum is the widest accumulator).
constexpr size_t SCRATCH_PARTIALS = 256;
constexpr size_t SCRATCH_BYTES = SCRATCH_PARTIALS + (size_t)MAX_BLOCKS * 16;
static_assert(SCRATCH_BYTES == APPFIS_NOALLOC_REDUCE_SCRATCH_BYTES, "header and kernel disagree on the scratch size");

// items is 0 for an empty box: one block then writes the identity
template <int V>
Split split_of(const Box& b)
{
    Split sp;
    sp.rows = (uint64_t)b.n1 * b.n2;
    sp.chunks = b.n0 > 0 ? (b.n0 - 1) / V + 1 : 0;
    sp.log_lanes = 0;
    while (sp.log_lanes < 6 && (1 << sp.log_lanes) < sp.chunks) sp.log_lanes++;
    const int lanes = 1 << sp.log_lanes;
    sp.segs = sp.chunks > 0 ? (sp.chunks - 1) / lanes + 1 : 0;
    const uint64_t per = 64 / lanes;
    sp.items = (sp.rows + per - 1) / per * sp.segs;
    return sp;
}

// scratch: SCRATCH_BYTES of device memory whose ticket word is zero at launch (the last
// block resets it, so consecutive reductions on one scratch need no clearing)
template <typename T, int OP, int V>
int launch_reduce(appfis_ctx* ctx, const void* data, const Box& b, void* dev_out, void* scratch)
{
    using A = typename Ops<T, OP>::A;
    const Split sp = split_of<V>(b);
    // A block's end costs about 20 ns of the launch (its ticket and fence are one after the
    // other): at most one block per CU, of 16 waves for boxes over 16 MB and of 4 below
    // (8192 x 8192 bytes: 256 blocks of 16 waves 22 us, 512 of 16 29 us, 1024 of 4 42 us, 256
    // of 4 38 us; 1024 x 1024 doubles: 256 of 4 11 us, 256 of 16 13 us, 1024 of 4 23 us).
    const unsigned threads = (double)sp.rows * b.n0 * sizeof(T) > (double)(16 << 20) ? MAX_RB : 256;
    // A wave takes U steps at once, except that up to 32 blocks are used to spread a small box
    // (80 x 96 doubles: 5.0 us as 20 blocks, 5.5 as 5).
    const uint64_t cap = ctx->num_cu > 0 && ctx->num_cu < MAX_BLOCKS ? ctx->num_cu : 256;
    const uint64_t waves = threads / 64, one = (sp.items + waves - 1) / waves, all = (one + U - 1) / U;
    const uint64_t want = std::min(cap, std::max(all, std::min<uint64_t>(one, 32)));
    const unsigned blocks = want < 1 ? 1u : (unsigned)want;
    if (SCRATCH_PARTIALS + (size_t)blocks * sizeof(A) > SCRATCH_BYTES)
        return invalid("reduce: %u partials exceed the %zu-byte scratch", blocks, SCRATCH_BYTES);
    unsigned* ticket = (unsigned*)scratch;
    A* partials = (A*)((char*)scratch + SCRATCH_PARTIALS);
    hipLaunchKernelGGL((k_reduce<T, OP, V>), dim3(blocks), dim3(threads), 0, ctx->stream, (const T*)data, b, sp, partials,
                       ticket, dev_out);
    APPFIS_LAUNCH_CHECK();
    return APPFIS_OK;
}

template <typename T, int OP>
int launch_rows(appfis_ctx* ctx, const void* data, const Box& b, void* dev_out, void* scratch)
{
    constexpr int V = 16 / (int)sizeof(T);
    return b.n0 >= V ? launch_reduce<T, OP, V>(ctx, data, b, dev_out, scratch)
                     : launch_reduce<T, OP, 1>(ctx, data, b, dev_out, scratch);
}

template <typename T>
int dispatch_op(appfis_ctx* ctx, const void* data, const Box& b, int op, void* dev_out, void* scratch)
{
    switch (op) {
    case APPFIS_MAX: return launch_rows<T, APPFIS_MAX>(ctx, data, b, dev_out, scratch);
    case APPFIS_MIN: return launch_rows<T, APPFIS_MIN>(ctx, data, b, dev_out, scratch);
    case APPFIS_SUM: return launch_rows<T, APPFIS_SUM>(ctx, data, b, dev_out, scratch);
    default: return invalid("unknown reduction op %d", op);
    }
}

int make_box(int ndim, const int* dims, const int* box, Box* b, uint64_t* n)
{
    int d[3];
    int st = check_shape(ndim, dims, d);
    if (st) return st;
    APPFIS_REQUIRE(box, "box is NULL");
    int s[3] = {0, 0, 0}, e[3] = {1, 1, 1};
    for (int a = 0; a < ndim; a++) {
        s[a] = box[2 * a];
        e[a] = box[2 * a + 1];
        APPFIS_REQUIRE(s[a] >= 0 && e[a] <= d[a], "box [%d,%d) outside dims[%d] = %d", s[a], e[a], a, d[a]);
    }
    b->d0 = d[0];
    b->d1 = d[1];
    b->s0 = s[0];
    b->s1 = s[1];
    b->s2 = s[2];
    b->n0 = e[0] > s[0] ? e[0] - s[0] : 0;
    b->n1 = e[1] > s[1] ? e[1] - s[1] : 0;
    b->n2 = e[2] > s[2] ? e[2] - s[2] : 0;
    *n = (uint64_t)b->n0 * b->n1 * b->n2;
    return APPFIS_OK;
}

int reduce_to_device(appfis_ctx* ctx, const void* data, int dtype, int ndim, const int* dims, const int* box, int op,
                     void* dev_out, void* scratch)
{
    Box b;
    uint64_t n;
    int st = make_box(ndim, dims, box, &b, &n);
    if (st) return st;
    if (n == 0) b.n0 = b.n1 = b.n2 = 0;  // empty box: kernel writes the identity
    switch (dtype) {
    case APPFIS_U8: return dispatch_op<uint8_t>(ctx, data, b, op, dev_out, scratch);
    case APPFIS_I32: return dispatch_op<int32_t>(ctx, data, b, op, dev_out, scratch);
    case APPFIS_F32: return dispatch_op<float>(ctx, data, b, op, dev_out, scratch);
    case APPFIS_F64: return dispatch_op<double>(ctx, data, b, op, dev_out, scratch);
    default: return invalid("reduce: unsupported dtype %d", dtype);
    }
}

// The context scratch of the allocating entry points.
int ctx_reduce_scratch(appfis_ctx* ctx, void** scratch)
{
    int st = ensure_scratch(ctx, SCRATCH_BYTES);
    if (st) return st;
    *scratch = ctx->scratch;
    return APPFIS_OK;
}

// A reduction whose 8-byte wide result the host waits for: the last block writes it into the
// context's pinned staging memory, which the GPU reaches directly, so that the call waits for
// one kernel and not for a copy of 8 bytes after it (a call on 80 x 96 doubles: 19 us against 27).
int reduce_to_host(appfis_ctx* ctx, const void* data, int dtype, int ndim, const int* dims, const int* box, int op,
                   void* wide)
{
    void* scr = nullptr;
    int st = ctx_reduce_scratch(ctx, &scr);
    if (st) return st;
    st = ensure_pinned(ctx, 8);
    if (st) return st;
    st = reduce_to_device(ctx, data, dtype, ndim, dims, box, op, ctx->pinned, scr);
    if (st) return st;
    APPFIS_HIP_CHECK(hipStreamSynchronize(ctx->stream));
    memcpy(wide, ctx->pinned, 8);
    return APPFIS_OK;
}

}  // namespace

// ---- fixed scratch of appfis_reduce_device_noalloc --------------------------------
// One copy per GPU, zero at module load and held until the process ends.  Host code
// never passes the symbol itself to a kernel (on the host it only names the variable):
// it passes the device address that hipGetSymbolAddress returned for the current GPU.
static __device__ __align__(256) unsigned char scratch[SCRATCH_BYTES];

namespace {

constexpr int MAX_DEVICES = 64;
std::mutex g_scratch_mutex;
void* g_scratch_ptr[MAX_DEVICES] = {};

__global__ void k_clear_ticket(unsigned* ticket) { *ticket = 0u; }

}  // namespace

namespace appfis {

int noalloc_scratch_setup(int device)
{
    if (device < 0 || device >= MAX_DEVICES)
        return invalid("device %d: the fixed reduction scratch supports devices 0..%d", device, MAX_DEVICES - 1);
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    if (g_scratch_ptr[device]) return APPFIS_OK;
    int cur = -1;
    APPFIS_HIP_CHECK(hipGetDevice(&cur));
    if (cur != device) return invalid("noalloc_scratch_setup: device %d is not current (%d is)", device, cur);
    void* ptr = nullptr;
    APPFIS_HIP_CHECK(hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)));
    if (!ptr) return invalid("hipGetSymbolAddress returned NULL for the reduction scratch");
    g_scratch_ptr[device] = ptr;
    return APPFIS_OK;
}

}  // namespace appfis

namespace {

void* noalloc_scratch(int device)
{
    if (device < 0 || device >= MAX_DEVICES) return nullptr;
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    return g_scratch_ptr[device];
}

}  // namespace

extern "C" {

int appfis_reduce_device(appfis_ctx* ctx, const void* data, int dtype, int ndim, const int* dims, const int* box,
                         int op, void* dev_result)
{
    APPFIS_REQUIRE(ctx && data && dev_result, "NULL argument");
    void* scr = nullptr;
    int st = ctx_reduce_scratch(ctx, &scr);
    if (st) return st;
    return reduce_to_device(ctx, data, dtype, ndim, dims, box, op, dev_result, scr);
}

int appfis_reduce_device_noalloc(appfis_ctx* ctx, const void* data, int dtype, int ndim, const int* dims,
                                 const int* box, int op, void* dev_result)
{
    APPFIS_REQUIRE(ctx && data && dev_result, "NULL argument");
    void* scr = noalloc_scratch(ctx->device);
    APPFIS_REQUIRE(scr, "device %d has no fixed reduction scratch (context not created through appfis_ctx_create)",
                   ctx->device);
    // the ticket must start at zero: a one-thread kernel clears it (a kernel, not a
    // memset node, so that the call can be captured into a graph)
    hipLaunchKernelGGL(k_clear_ticket, dim3(1), dim3(1), 0, ctx->stream, (unsigned*)scr);
    APPFIS_LAUNCH_CHECK();
    return reduce_to_device(ctx, data, dtype, ndim, dims, box, op, dev_result, scr);
}

int appfis_reduce_sum_wide(appfis_ctx* ctx, const void* data, int dtype, int ndim, const int* dims, const int* box,
                           void* result)
{
    APPFIS_REQUIRE(ctx && data && result, "NULL argument");
    APPFIS_NOT_CAPTURING(ctx, "a reduction with a host result (use appfis_reduce_device)");
    return reduce_to_host(ctx, data, dtype, ndim, dims, box, APPFIS_SUM, result);
}

int appfis_reduce(appfis_ctx* ctx, const void* data, int dtype, int ndim, const int* dims, const int* box, int op,
                  void* result)
{
    APPFIS_REQUIRE(ctx && data && result, "NULL argument");
    APPFIS_NOT_CAPTURING(ctx, "a reduction with a host result (use appfis_reduce_device)");
    unsigned char wide[8];
    const int st = reduce_to_host(ctx, data, dtype, ndim, dims, box, op, wide);
    if (st) return st;
    size_t es = dtype_size(dtype);
    if (op != APPFIS_SUM) {
        memcpy(result, wide, es);
        return APPFIS_OK;
    }
    // SUM: round the widened result to T once
    if (dtype == APPFIS_U8 || dtype == APPFIS_I32) {
        long long v;
        memcpy(&v, wide, 8);
        if (dtype == APPFIS_U8) *(uint8_t*)result = (uint8_t)v;
        else *(int32_t*)result = (int32_t)v;
    } else {
        double v;
        memcpy(&v, wide, 8);
        if (dtype == APPFIS_F32) *(float*)result = (float)v;
        else *(double*)result = v;
    }
    return APPFIS_OK;
}

}  // extern "C"
