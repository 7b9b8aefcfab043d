// HeatDiffusion 2D 5-point explicit sweep (config form of the reference functor
// HeatDiffusion/src/heat_appfis.hpp:166-174, driven like heat_appfis.hpp:86-91 on a
// DUAL grid: sweep, then Grid::Swap).
//
//   u' = u + c*((((uN + uS) + uE) + uW) - 4u)      each operation rounded
//
// PLAIN : one sweep per launch, one output per thread, x along the wave.
// CHOSEN: temporal blocking.  A block loads a window of the field with a T-cell halo into
//         registers and advances it T sweeps there, then writes the window's centre; the
//         valid region shrinks by one cell per sweep (k_heat2d_rt; k_heat2d_whole is the
//         window that holds a whole small grid and needs no halo).  Dirichlet ghost cells
//         are loaded and never updated, exactly as in the one-sweep form, so every interior
//         value is bit-identical to PLAIN.  HBM/MALL traffic per sweep drops by ~T.
#include "common.hpp"

#include <algorithm>
#include <cmath>
#include <type_traits>
#include <vector>

using namespace appfis;

namespace {

// One sweep; a thread owns RY consecutive rows of one column, so the column's RY+2
// values are loaded once and its loads are all in flight together.  Block 64 x 4
// threads = a 64 x 4*RY tile; tiles are spread over the XCDs in contiguous runs.
template <typename T, int RY>
__global__ __launch_bounds__(256) void k_heat2d_plain(const T* __restrict__ u, T* __restrict__ v, int nx, int ny,
                                                      T c)
{
    const int W = nx + 2;
    const unsigned gx = gridDim.x;
    const unsigned t = xcd_tile(blockIdx.x + gx * blockIdx.y, gx * gridDim.y);
    const int i = (int)(t % gx) * 64 + threadIdx.x + 1;
    const int j0 = ((int)(t / gx) * 4 + threadIdx.y) * RY + 1;
    if (i > nx || j0 > ny) return;
    T col[RY + 2], e[RY], w[RY];
#pragma unroll
    for (int r = 0; r < RY + 2; r++) {
        const int j = j0 - 1 + r;
        col[r] = j <= ny + 1 ? u[i + (size_t)W * j] : (T)0;
    }
#pragma unroll
    for (int r = 0; r < RY; r++) {
        const size_t o = i + (size_t)W * (j0 + r);
        e[r] = j0 + r <= ny ? u[o + 1] : (T)0;
        w[r] = j0 + r <= ny ? u[o - 1] : (T)0;
    }
#pragma unroll
    for (int r = 0; r < RY; r++) {
        if (j0 + r > ny) break;
        const T uc = col[r + 1];
        T s = col[r] + col[r + 2];
        s = s + e[r];
        s = s + w[r];
        s = s - (T)4 * uc;
        v[i + (size_t)W * (j0 + r)] = uc + c * s;
    }
}

// Ensemble: grid s owns tiles tile0 .. tile0 + tiles_x * tiles_y - 1 of one launch.
template <typename T>
struct HeatGrid {
    T* b[2];
    int nx, ny, tiles_x, tile0;
};

// The grid that owns tile `tile` of an ensemble launch: binary search over tile0 (the
// same for every thread of the block).
template <typename T>
__device__ inline int grid_of_tile(const HeatGrid<T>* __restrict__ tab, int ngrid, int tile)
{
    int lo = 0, hi = ngrid - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (tab[mid].tile0 <= tile) lo = mid;
        else hi = mid - 1;
    }
    return lo;
}

// Register tiles: a block of NW waves holds a window of 64*WPL columns x NW*K rows, lane
// l owning columns WPL*l .. WPL*l+WPL-1 of K consecutive rows (wave w: window rows w*K ..
// w*K+K-1) in registers.  A sweep takes a cell's east / west neighbours from the lane's
// own registers, or by DPP from lanes l+1 / l-1 for its outer columns, and the north /
// south ones from the lane's own registers; only each wave's first and last rows go
// through LDS, in two slots alternating with the sweep's parity, so a sweep has one
// barrier.  Cells at the window's edge read meaningless neighbours (zero from the DPP
// shift at lanes 0 / 63, the wave's own edge rows above the first wave and below the
// last), which spoils one more ring per sweep; after TS sweeps the centre
// (64*WPL-2TS) x (NW*K-2TS) is exact.  Ghost cells keep their loaded values, so every
// interior value equals the one-sweep form's.
//
// The adds and multiplies bound it, so a cell does no more of anything than it needs: a block whose
// window is all interior skips the selects, and rt_tile is forced inline (as a call, which two
// callers made of it, the cells went through the calling convention's registers and scratch:
// 120 registers for 7 x 1 cells, 53 inlined).  Further, 1024^2 on 256 CUs, us per sweep, the
// 96 x 48 tile of 16 sweeps:
//   FP64: sum - 4u as one FMA, 1.24 -> 1.20 (of these 0.02 are the check).  4u is exact where it
//   does not overflow, so the FMA then rounds as the subtraction does.  `big` is the top word of a
//   magnitude that the launch's sweeps cannot grow that far from; a block that loaded a larger one,
//   an infinity or a NaN does its sweeps again with a multiply and a subtraction.  That loop is
//   short and out of the way: a launch fetches its code anew (0.7 us a launch less than with
//   two sweeps a trip in line).
//   FP32: a row's update starts when the row two above it is done (an empty asm that takes both),
//   which keeps the schedule from stretching over the whole column of rows: 0.889 -> 0.868, and
//   2048^2 2.035 -> 1.978.  In FP64 the same costs 1 %, and the FMA's check costs FP32 5 %.
template <typename T, int K, int NW, int TS, int WPL, bool WHOLE>
__device__ __forceinline__ void rt_tile(const T* __restrict__ u, T* __restrict__ v, int nx, int ny, T c, int steps,
                               unsigned big, int tbx, int tby)
{
    constexpr int TX = 64 * WPL - 2 * TS, TY = NW * K - 2 * TS;
    static_assert(WHOLE || (TX > 0 && TY > 0), "the window must be wider and taller than its halo");
    __shared__ T edge[2][NW][2][WPL][64];
    constexpr bool kFused = sizeof(T) == 8;
    __shared__ int large[kFused ? NW : 1];
    const gmem<T>* ug = to_global(u);  // the ensemble reads u and v from its grid table
    gmem<T>* vg = to_global(v);
    const int W = nx + 2, H = ny + 2;
    const int lane = (int)(threadIdx.x & 63);
    const int wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int wx0 = WHOLE ? 0 : tbx * TX + 1 - TS;  // padded column and row of the window
    const int wy0 = WHOLE ? 0 : tby * TY + 1 - TS;
    const int gx0 = wx0 + WPL * lane;  // of R[.][0]
    const int gy0 = wy0 + wv * K;      // of R[0][.]
    bool col_in[WPL];
#pragma unroll
    for (int w = 0; w < WPL; w++) col_in[w] = gx0 + w >= 1 && gx0 + w <= nx;
    T R[K][WPL];
    auto load = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int k = 0; k < K; k++) {
            const int gy = gy0 + k;
#pragma unroll
            for (int w = 0; w < WPL; w++) {
                const int gx = gx0 + w;
                R[k][w] = (gx >= 0 && gx < W && gy >= 0 && gy < H) ? ug[(size_t)gx + (size_t)W * (size_t)gy] : (T)0;
            }
        }
    };
    load();
    // one sweep; its edge rows use LDS slot b (sweeps alternate slots)
    auto sweep = [&](auto masked, auto fused, const int b) __attribute__((always_inline)) {
#pragma unroll
        for (int w = 0; w < WPL; w++) {
            edge[b][wv][0][w][lane] = R[0][w];
            edge[b][wv][1][w][lane] = R[K - 1][w];
        }
        __syncthreads();
        // the row above row k before this sweep, and the row below the wave.  The block's
        // first and last waves read their own slots instead: rows outside the window only
        // reach the halo ring, which is never stored.
        const int wu = wv > 0 ? wv - 1 : wv, wd = wv < NW - 1 ? wv + 1 : wv;
        T above[WPL], dn[WPL];
#pragma unroll
        for (int w = 0; w < WPL; w++) {
            above[w] = edge[b][wu][1][w][lane];
            dn[w] = edge[b][wd][0][w][lane];
        }
#pragma unroll
        for (int k = 0; k < K; k++) {
            const T east = lane_shift_z<false>(R[k][0]);       // lane l+1's first column
            const T west = lane_shift_z<true>(R[k][WPL - 1]);  // lane l-1's last column
            const int gy = gy0 + k;
            const bool row_in = gy >= 1 && gy <= ny;
            T nv[WPL];
#pragma unroll
            for (int w = 0; w < WPL; w++) {
                const T uc = R[k][w];
                T sum = above[w] + (k == K - 1 ? dn[w] : R[k + 1][w]);
                sum = sum + (w == WPL - 1 ? east : R[k][w + 1]);
                sum = sum + (w == 0 ? west : R[k][w - 1]);
                if constexpr (decltype(fused)::value) sum = __builtin_elementwise_fma((T)-4, uc, sum);
                else sum = sum - (T)4 * uc;
                const T next = uc + c * sum;
                nv[w] = !decltype(masked)::value || (col_in[w] && row_in) ? next : uc;
            }
#pragma unroll
            for (int w = 0; w < WPL; w++) {
                above[w] = R[k][w];
                R[k][w] = nv[w];
            }
            // FP32 only (see above): row k + 2 waits for row k
            if constexpr (!kFused)
                if (k + 2 < K)
#pragma unroll
                    for (int w = 0; w < WPL; w++) asm volatile("" : "+v"(R[k + 2][w]) : "v"(nv[w]));
        }
    };
    // two sweeps per trip, so that the registers of consecutive sweeps are renamed
    // rather than copied
    auto sweeps = [&](auto masked, auto fused) __attribute__((always_inline)) {
        for (int s = 0; s + 1 < steps; s += 2) {
            sweep(masked, fused, 0);
            sweep(masked, fused, 1);
        }
        if (steps & 1) sweep(masked, fused, 0);
    };
    if constexpr (kFused) {
        unsigned top = 0;
#pragma unroll
        for (int k = 0; k < K; k++)
#pragma unroll
            for (int w = 0; w < WPL; w++) top = max(top, (unsigned)__double2hiint(R[k][w]) & 0x7fffffffu);
        const bool wave_large = __any(top >= big);
        if (lane == 0) large[wv] = wave_large;  // read after the sweeps: their barriers order it
    }
    const bool inner = wx0 >= 1 && wx0 + 64 * WPL - 1 <= nx && wy0 >= 1 && wy0 + NW * K - 1 <= ny;
    if (inner) sweeps(std::false_type{}, std::bool_constant<kFused>{});
    else sweeps(std::true_type{}, std::bool_constant<kFused>{});
    if constexpr (kFused)
        if (__builtin_expect(__any(large[lane % NW]), 0)) {
            __syncthreads();  // the last sweep's edge rows have been read
            load();
#pragma clang loop unroll(disable)
            for (int s = 0; s < steps; s++) sweep(std::true_type{}, std::false_type{}, s & 1);
        }
    // the centre: window columns TS .. TS+TX-1, rows TS .. TS+TY-1 (interior cells only).  The
    // column is made opaque: the loads' addresses would be kept in registers for the stores.
    int sx0 = gx0;
    asm volatile("" : "+v"(sx0));
#pragma unroll
    for (int k = 0; k < K; k++) {
        const int r = wv * K + k, gy = gy0 + k;
        if ((!WHOLE && (r < TS || r >= TS + TY)) || gy < 1 || gy > ny) continue;
#pragma unroll
        for (int w = 0; w < WPL; w++) {
            const int lx = WPL * lane + w;
            if ((WHOLE || (lx >= TS && lx < TS + TX)) && sx0 + w >= 1 && sx0 + w <= nx)
                vg[(size_t)(sx0 + w) + (size_t)W * (size_t)gy] = R[k][w];
        }
    }
}

template <typename T, int K, int NW, int TS, int WPL>
__global__ __launch_bounds__(64 * NW) void k_heat2d_rt(const T* __restrict__ u, T* __restrict__ v, int nx, int ny,
                                                       T c, int steps, unsigned big)
{
    constexpr int TX = 64 * WPL - 2 * TS;
    const int tiles_x = (nx + TX - 1) / TX;
    const int t = (int)xcd_tile(blockIdx.x, gridDim.x);
    const int tby = t / tiles_x;
    rt_tile<T, K, NW, TS, WPL, false>(u, v, nx, ny, c, steps, big, t - tby * tiles_x, tby);
}

// A grid that fits one block's window, ghost ring included, needs no halo: its cells at the
// window's edge are ghost cells, which keep their values, so one launch of one block runs as many
// sweeps as it is given.
template <typename T, int K, int NW, int WPL>
__global__ __launch_bounds__(64 * NW) void k_heat2d_whole(const T* __restrict__ u, T* __restrict__ v, int nx, int ny,
                                                          T c, int steps, unsigned big)
{
    rt_tile<T, K, NW, 0, WPL, true>(u, v, nx, ny, c, steps, big, 0, 0);
}

template <typename T, int K, int NW, int TS, int WPL>
__global__ __launch_bounds__(64 * NW) void k_heat2d_rt_ens(const HeatGrid<T>* __restrict__ tab, int ngrid, int par,
                                                           T c, int steps, unsigned big)
{
    const int tile = (int)xcd_tile(blockIdx.x, gridDim.x);
    const HeatGrid<T>& G = tab[grid_of_tile(tab, ngrid, tile)];
    const int t = tile - G.tile0;
    const int tby = t / G.tiles_x;
    rt_tile<T, K, NW, TS, WPL, false>(G.b[par], G.b[par ^ 1], G.nx, G.ny, c, steps, big, t - tby * G.tiles_x, tby);
}

constexpr int PLAIN_RY = 4;

template <typename T>
int run_plain(appfis_ctx* ctx, T* b0, T* b1, int nx, int ny, T c, int iters)
{
    dim3 block(64, 4), grid(ceil_div(nx, 64), ceil_div(ny, 4 * PLAIN_RY));
    T* buf[2] = {b0, b1};
    for (int it = 0; it < iters; it++) {
        hipLaunchKernelGGL((k_heat2d_plain<T, PLAIN_RY>), grid, block, 0, ctx->stream, buf[it & 1],
                           buf[(it + 1) & 1], nx, ny, c);
        APPFIS_LAUNCH_CHECK();
    }
    return APPFIS_OK;
}

// Split `iters` sweeps into launches of at most TS sweeps such that the number of
// launches has the parity of `iters`: the field then ends in bufs[iters % 2], as
// with one sweep per launch.
inline int launch_count(int iters, int ts)
{
    int n = (iters + ts - 1) / ts;
    if ((n & 1) != (iters & 1)) n++;
    return n > iters ? iters : n;
}

inline int plan_launches(int iters, int ts, int* counts, int max_launches)
{
    const int n = launch_count(iters, ts);
    if (n > max_launches) return -1;
    int base = iters / n, extra = iters % n;
    for (int l = 0; l < n; l++) counts[l] = base + (l < extra ? 1 : 0);
    return n;
}

// The top word of an FP64 magnitude below which all stay under a quarter of the largest double
// through `steps` sweeps: a sweep multiplies the largest magnitude by at most |1 - 4c| + 4|c|
// and its roundings.  0 (no magnitude is below it) where there is none.
inline unsigned fused_limit(double c, int steps)
{
    const double e = 1020.0 - steps * (std::log2(std::fabs(1.0 - 4.0 * c) + 4.0 * std::fabs(c)) + 1e-9);
    return e > -1000.0 ? (unsigned)(1023 + (int)std::floor(e)) << 20 : 0;
}

template <typename T, int K, int NW, int TS, int WPL>
int run_rt(appfis_ctx* ctx, void* b0, void* b1, int nx, int ny, double c, int iters, int depth)
{
    constexpr int TX = 64 * WPL - 2 * TS, TY = NW * K - 2 * TS;
    T* buf[2] = {(T*)b0, (T*)b1};
    const size_t tiles = (size_t)ceil_div(nx, TX) * ceil_div(ny, TY);
    APPFIS_REQUIRE(tiles < (1u << 31), "heat2d: too many tiles");
    std::vector<int> counts((size_t)iters);
    int n = plan_launches(iters, depth < TS ? depth : TS, counts.data(), iters);
    if (n <= 0) return invalid("heat2d: cannot split %d sweeps", iters);
    for (int l = 0; l < n; l++) {
        hipLaunchKernelGGL((k_heat2d_rt<T, K, NW, TS, WPL>), dim3((unsigned)tiles), dim3(64 * NW), 0, ctx->stream,
                           buf[l & 1], buf[(l + 1) & 1], nx, ny, (T)c, counts[l],
                           fused_limit(c, counts[l]));
        APPFIS_LAUNCH_CHECK();
    }
    return APPFIS_OK;
}

// Grids that fit the window of one block with K rows in each of NW waves.
template <int K, int NW, int WPL>
constexpr bool whole_fits(int nx, int ny)
{
    return nx <= 64 * WPL - 2 && ny <= NW * K - 2;
}

// The whole grid in one block where it fits; else the first tiles of the tables below.
template <typename T, int K, int NW, int WPL>
int run_whole(appfis_ctx* ctx, void* b0, void* b1, int nx, int ny, double c, int iters, int)
{
    if (!whole_fits<K, NW, WPL>(nx, ny)) return run_rt<T, 8, 8, 8, 1>(ctx, b0, b1, nx, ny, c, iters, 8);
    T* buf[2] = {(T*)b0, (T*)b1};
    const int n = launch_count(iters, 1024);  // a launch ends within a millisecond or so
    for (int l = 0; l < n; l++) {
        const int steps = iters / n + (l < iters % n ? 1 : 0);
        hipLaunchKernelGGL((k_heat2d_whole<T, K, NW, WPL>), dim3(1), dim3(64 * NW), 0, ctx->stream, buf[l & 1],
                           buf[(l + 1) & 1], nx, ny, (T)c, steps, fused_limit(c, steps));
        APPFIS_LAUNCH_CHECK();
    }
    return APPFIS_OK;
}

struct HeatVariant {
    const char* name;
    int (*fn)(appfis_ctx*, void*, void*, int, int, double, int, int);
    int ts;  // sweeps per launch at most
};

// Temporal-blocking candidates (output tile TX x TY, TS sweeps per launch, K rows in each of NW
// waves; "rt2": two columns per lane).  A launch costs about 5 us before its first sweep's worth of
// work, and tiles load and compute a halo of TS cells around their output: the deepest are best
// while the tiles fit the CUs about once, in the smallest window that makes it so (FP64, us per
// sweep: 96 x 80 32x16 0.84, 48x24 1.03; 512^2 32x32 0.78, 48x24 0.87, 96x48 1.19; 1024^2 96x48
// 1.20, 48x48 1.32).  Beyond that the adds decide (4096^2: 48x96 k14 10.3, k7 14.5, 96x48 over
// 12.2).  "whole" needs no halo, but one CU does all the work: 62^2 takes 0.82, 48 x 48 the
// same and in 32x16 tiles 0.83.  A fixed depth takes the first entry that holds it.
template <typename T>
static const HeatVariant kHeat[] = {
    {"rt 48x48 ts8 k8 w8", run_rt<T, 8, 8, 8, 1>, 8},
    {"rt 48x96 ts8 k7 w16", run_rt<T, 7, 16, 8, 1>, 8},
    {"rt 48x96 ts8 k14 w8", run_rt<T, 14, 8, 8, 1>, 8},
    {"rt 48x24 ts8 k5 w8", run_rt<T, 5, 8, 8, 1>, 8},
    {"rt 48x32 ts8 k6 w8", run_rt<T, 6, 8, 8, 1>, 8},
    {"rt 48x48 ts8 k4 w16", run_rt<T, 4, 16, 8, 1>, 8},
    {"rt2 112x48 ts8 k8 w8", run_rt<T, 8, 8, 8, 2>, 8},
    {"rt 40x72 ts12 k12 w8", run_rt<T, 12, 8, 12, 1>, 12},
    {"rt2 104x56 ts12 k5 w16", run_rt<T, 5, 16, 12, 2>, 12},
    {"rt2 96x48 ts16 k5 w16", run_rt<T, 5, 16, 16, 2>, 16},
    {"rt 32x16 ts16 k6 w8", run_rt<T, 6, 8, 16, 1>, 16},
    {"rt 32x32 ts16 k4 w16", run_rt<T, 4, 16, 16, 1>, 16},
    {"whole 64x80 k5 w16", run_whole<T, 5, 16, 1>, 0},
};
constexpr int SHALLOW = 8;
constexpr int kHeatCount = (int)(sizeof(kHeat<double>) / sizeof(kHeat<double>[0]));

}  // namespace

extern "C" int appfis_heat2d(appfis_ctx* ctx, int dtype, void* buf0, void* buf1, int nx, int ny, double c, int iters,
                             int variant, int tsteps)
{
    APPFIS_REQUIRE(ctx && buf0 && buf1, "NULL argument");
    APPFIS_REQUIRE(nx > 0 && ny > 0, "interior must be non-empty (nx=%d ny=%d)", nx, ny);
    APPFIS_REQUIRE((double)(nx + 2) * (ny + 2) < 2147483647.0, "grid exceeds the int index range");
    APPFIS_REQUIRE(iters >= 0, "iters must be >= 0");
    APPFIS_REQUIRE(buf0 != buf1, "the two buffers must differ");
    if (iters == 0) return APPFIS_OK;
    if (variant == APPFIS_PLAIN) {
        if (dtype == APPFIS_F64) return run_plain<double>(ctx, (double*)buf0, (double*)buf1, nx, ny, c, iters);
        if (dtype == APPFIS_F32) return run_plain<float>(ctx, (float*)buf0, (float*)buf1, nx, ny, (float)c, iters);
        return invalid("heat2d: dtype must be F64 or F32");
    }
    if (variant == APPFIS_CHOSEN) {
        if (dtype != APPFIS_F64 && dtype != APPFIS_F32) return invalid("heat2d: dtype must be F64 or F32");
        const HeatVariant* tab = dtype == APPFIS_F64 ? kHeat<double> : kHeat<float>;
        if (tsteps > 0) {
            // caller-fixed depth: the first candidate that holds that many sweeps per launch
            for (int i = 0; i < kHeatCount; i++)
                if (tab[i].ts >= tsteps) return tab[i].fn(ctx, buf0, buf1, nx, ny, c, iters, tsteps);
            return invalid("heat2d: tsteps %d exceeds the deepest temporal blocking (16)", tsteps);
        }
        // autotuned tile shape and depth, timed once per shape on scratch buffers over 96 sweeps
        // (an even number of full launches at depths 8, 12 and 16 alike); every
        // candidate computes the same values in the same order
        const int key[6] = {1, dtype, nx, ny, 0, 0};
        if (!tuned_entry(ctx, key)) {
            APPFIS_NOT_CAPTURING(ctx, "appfis_heat2d CHOSEN's first call for a shape (autotuning)");
            const size_t half = ((size_t)(nx + 2) * (ny + 2) * dtype_size(dtype) + 255) / 256 * 256;
            int st = ensure_work(ctx, 2 * half);
            if (st) return st;
            void* const s0 = ctx->work;
            void* const s1 = (char*)ctx->work + half;
            APPFIS_HIP_CHECK(hipMemsetAsync(ctx->work, 0, 2 * half, ctx->stream));
            // every candidate that differs here: "whole", the last, only where the grid fits it
            const int ntab = whole_fits<5, 16, 1>(nx, ny) ? kHeatCount : kHeatCount - 1;
            std::vector<const char*> names;
            for (int i = 0; i < ntab; i++) names.push_back(tab[i].name);
            int pick = 0;
            st = tune_select(ctx, key, ntab, names.data(),
                             [&](int i) { return tab[i].fn(ctx, s0, s1, nx, ny, c, 96, tab[i].ts); }, 3, &pick);
            if (st) return st;
            appfis_tune_entry& e = ctx->tuned.back();
            for (int i = 0; i < ntab; i++)
                if (tab[i].ts == SHALLOW && (tab[e.param].ts != SHALLOW || e.ms[i] < e.ms[e.param])) e.param = i;
        }
        // The launches of a call have the parity of its sweeps, so calls of one and two take one
        // launch a sweep in any form, and PLAIN's needs no halo (us, tiles / PLAIN: 2048^2 FP32
        // 12.5 / 8.0, 1000^2 FP64 6.1 / 4.8, 8192^2 FP64 277 / 239).  Where the deep tiles' halo
        // saves no launch the best shallow ones are faster (1000^2 FP64, 5 sweeps 9.5 / 8.3, 16
        // sweeps 23.9 / 20.5, 20 sweeps 27.0 / 32.7; 96 x 80, 7 sweeps 5.6 / 5.0).
        if (iters <= 2)
            return dtype == APPFIS_F64 ? run_plain<double>(ctx, (double*)buf0, (double*)buf1, nx, ny, c, iters)
                                       : run_plain<float>(ctx, (float*)buf0, (float*)buf1, nx, ny, (float)c, iters);
        const appfis_tune_entry* e = tuned_entry(ctx, key);
        const int ts = tab[e->choice].ts;
        const bool shallow = ts > SHALLOW && launch_count(iters, SHALLOW) == launch_count(iters, ts);
        const HeatVariant& v = tab[shallow ? e->param : e->choice];
        return v.fn(ctx, buf0, buf1, nx, ny, c, iters, v.ts);
    }
    if (variant >= APPFIS_CANDIDATE0) {
        if (dtype != APPFIS_F64 && dtype != APPFIS_F32) return invalid("heat2d: dtype must be F64 or F32");
        const HeatVariant* tab = dtype == APPFIS_F64 ? kHeat<double> : kHeat<float>;
        const int i = variant - APPFIS_CANDIDATE0;
        APPFIS_REQUIRE(i < kHeatCount, "heat2d: candidate %d out of range (%d candidates)", i, kHeatCount);
        return tab[i].fn(ctx, buf0, buf1, nx, ny, c, iters, tab[i].ts);
    }
    return invalid("heat2d: unknown variant %d", variant);
}

// Ensemble launches of the register tiles, at most TS sweeps each.
template <typename T, int K, int NW, int TS, int WPL>
int run_ensemble(appfis_ctx* ctx, int ngrid, const int* nx, const int* ny, void* const* buf0,
                 void* const* buf1, double c, int iters)
{
    constexpr int TX = 64 * WPL - 2 * TS, TY = NW * K - 2 * TS;
    const auto kern = k_heat2d_rt_ens<T, K, NW, TS, WPL>;
    std::vector<HeatGrid<T>> hg((size_t)ngrid);
    long long tiles = 0;
    for (int g = 0; g < ngrid; g++) {
        APPFIS_REQUIRE(nx[g] > 0 && ny[g] > 0, "heat2d ensemble: grid %d is empty", g);
        APPFIS_REQUIRE((double)(nx[g] + 2) * (ny[g] + 2) < 2147483647.0, "grid %d exceeds the int index range", g);
        APPFIS_REQUIRE(buf0[g] && buf1[g] && buf0[g] != buf1[g], "heat2d ensemble: grid %d buffers", g);
        hg[g].b[0] = (T*)buf0[g];
        hg[g].b[1] = (T*)buf1[g];
        hg[g].nx = nx[g];
        hg[g].ny = ny[g];
        hg[g].tiles_x = (int)ceil_div(nx[g], TX);
        hg[g].tile0 = (int)tiles;
        tiles += (long long)hg[g].tiles_x * ceil_div(ny[g], TY);
    }
    APPFIS_REQUIRE(tiles < (1LL << 31), "heat2d ensemble: too many tiles");
    const size_t tab_bytes = (size_t)ngrid * sizeof(HeatGrid<T>);
    int st = ensure_work(ctx, tab_bytes);
    if (st) return st;
    HeatGrid<T>* tab = (HeatGrid<T>*)ctx->work;
    APPFIS_HIP_CHECK(hipMemcpyAsync(tab, hg.data(), tab_bytes, hipMemcpyHostToDevice, ctx->stream));
    APPFIS_HIP_CHECK(hipStreamSynchronize(ctx->stream));  // the host table is a local
    std::vector<int> counts((size_t)iters);
    const int n = plan_launches(iters, TS, counts.data(), iters);
    if (n <= 0) return invalid("heat2d: cannot split %d sweeps", iters);
    // the whole launch chain is one graph, captured on the first call with these
    // arguments and replayed by later ones (it reads the grids from the table)
    const std::vector<uint64_t> key = {1, key_ptr((const void*)kern), key_ptr(tab), (uint64_t)ngrid,
                                       (uint64_t)tiles, key_bits(c), (uint64_t)iters};
    hipGraphExec_t exec = nullptr;
    st = cached_graph(ctx, key,
                      [&]() {
                          for (int l = 0; l < n; l++) {
                              hipLaunchKernelGGL(kern, dim3((unsigned)tiles), dim3(64 * NW), 0, ctx->stream, tab, ngrid,
                                                 l & 1, (T)c, counts[l], fused_limit(c, counts[l]));
                              APPFIS_LAUNCH_CHECK();
                          }
                          return APPFIS_OK;
                      },
                      &exec);
    if (st) return st;
    APPFIS_HIP_CHECK(hipGraphLaunch(exec, ctx->stream));
    // the table stays in use until the graph ran: wait before the workspace can be reused
    APPFIS_HIP_CHECK(hipStreamSynchronize(ctx->stream));
    return APPFIS_OK;
}

// Tiles an ensemble may take.  Its launches take about
//     launches * (launch + load * blocks per CU) + sweeps * sweep * blocks per CU
// us, `load` a block's window in and its tile out, blocks per CU being the mean of their number and
// of it rounded up, and at least a quarter: the tiles are those of the least sum.  The constants are
// fitted to 14 ensembles of 1 to 256 grids of 20 to 8192 cells a side and 1 to 200 sweeps; the choice
// is within 1 % of the best of the four on average, 10 % at most.  (Us for all sweeps, in the order
// below; FP64: two of 4000 x 4000 1 sweep 164, 146, 260, 182, 5 165, 161, 333, 251, 100 1878, 2356,
// 4173, 2816; 30 up to 256 10 sweeps 58, 58, 70, 61, 100 183, 181, 223, 159.  FP32: 64 of 64 to 883 x 137
// to 200 4 sweeps 78, 93, 140, 89, 100 343, 408, 613, 376.)
struct HeatEnsemble {
    int (*fn)(appfis_ctx*, int, const int*, const int*, void* const*, void* const*, double, int);
    int tx, ty, ts;
    double launch, load, sweep;
};
template <typename T, int K, int NW, int TS, int WPL>
constexpr HeatEnsemble ensemble_tiles(double launch, double load, double sweep)
{
    return {run_ensemble<T, K, NW, TS, WPL>, 64 * WPL - 2 * TS, NW * K - 2 * TS, TS, launch, load, sweep};
}
static const HeatEnsemble kEnsembleF64[] = {
    ensemble_tiles<double, 8, 8, 8, 2>(4.58, 4.12, 0.21),
    ensemble_tiles<double, 6, 8, 8, 1>(4.34, 1.05, 0.12),
    ensemble_tiles<double, 4, 16, 16, 1>(5.26, 1.42, 0.23),
    ensemble_tiles<double, 5, 16, 16, 2>(3.6, 3.97, 0.68),
};
static const HeatEnsemble kEnsembleF32[] = {
    ensemble_tiles<float, 8, 8, 8, 2>(5.04, 1.64, 0.19),
    ensemble_tiles<float, 6, 8, 8, 1>(4.09, 0.96, 0.05),
    ensemble_tiles<float, 4, 16, 16, 1>(4.51, 1.42, 0.12),
    ensemble_tiles<float, 5, 16, 16, 2>(5.69, 1.92, 0.3),
};

const HeatEnsemble& pick_ensemble(const HeatEnsemble (&tab)[4], int num_cu, int ngrid, const int* nx, const int* ny,
                                  int iters)
{
    int best = 0;
    double least = 0.0;
    for (int i = 0; i < 4; i++) {
        const HeatEnsemble& e = tab[i];
        double blocks = 0.0;
        for (int g = 0; g < ngrid; g++)
            if (nx[g] > 0 && ny[g] > 0) blocks += (double)ceil_div(nx[g], e.tx) * ceil_div(ny[g], e.ty);
        const double mean = blocks / (num_cu > 0 ? num_cu : 256), per_cu = std::max(0.5 * (mean + std::ceil(mean)), 0.25);
        const double cost = launch_count(iters, e.ts) * (e.launch + e.load * per_cu) + iters * e.sweep * per_cu;
        if (i == 0 || cost < least) {
            least = cost;
            best = i;
        }
    }
    return tab[best];
}

extern "C" int appfis_heat2d_ensemble(appfis_ctx* ctx, int dtype, int ngrid, const int* nx, const int* ny,
                                      void* const* buf0, void* const* buf1, double c, int iters)
{
    APPFIS_REQUIRE(ctx && nx && ny && buf0 && buf1, "NULL argument");
    APPFIS_NOT_CAPTURING(ctx, "appfis_heat2d_ensemble (it captures and replays a graph of its own)");
    APPFIS_REQUIRE(ngrid >= 1, "heat2d ensemble: need at least one grid");
    APPFIS_REQUIRE(iters >= 0, "iters must be >= 0");
    if (iters == 0) return APPFIS_OK;
    if (dtype == APPFIS_F64)
        return pick_ensemble(kEnsembleF64, ctx->num_cu, ngrid, nx, ny, iters).fn(ctx, ngrid, nx, ny, buf0, buf1, c, iters);
    if (dtype == APPFIS_F32)
        return pick_ensemble(kEnsembleF32, ctx->num_cu, ngrid, nx, ny, iters).fn(ctx, ngrid, nx, ny, buf0, buf1, c, iters);
    return invalid("heat2d ensemble: dtype must be F64 or F32");
}

extern "C" int appfis_heat2d_candidates(int dtype, char* names, int len)
{
    if (dtype != APPFIS_F64 && dtype != APPFIS_F32) return -invalid("heat2d: dtype must be F64 or F32");
    const HeatVariant* tab = dtype == APPFIS_F64 ? kHeat<double> : kHeat<float>;
    std::string all;
    for (int i = 0; i < kHeatCount; i++) all += std::string(tab[i].name) + "\n";
    if (names && len > 0) snprintf(names, (size_t)len, "%s", all.c_str());
    return kHeatCount;
}
