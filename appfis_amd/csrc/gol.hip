// GameOfLife 2D, uint8 cells, periodic, rule B3/S23 -- config form of the reference
// functor GameOfLife/src/game_appfis.hpp:121-135 driven on a periodic DUAL grid, where
// every generation is followed by the single-rank Exchange of the written buffer
// (Communication.hpp:613-678, X then Y over the full extents, so corners wrap).
//
// PLAIN: one generation per launch.  Each lane owns one CHUNK-byte (16) aligned chunk
//   of the padded buffer viewed as a linear byte array (rows are W = nx+2 bytes, so
//   chunks do not align with rows).  For a chunk whose cells lie in interior rows the
//   three input rows are p-W, p, p+W: the centre row is the aligned chunk itself, the
//   rows above and below are funnel-shifted out of aligned 16-byte loads by the
//   compile-time byte offset W mod 16 (one kernel instance per residue).  Neighbour
//   counts are SWAR byte sums (column sums, then +/-1 byte shifts with v_alignbyte),
//   the B3/S23 rule is a zero-byte test, and the chunk is stored with 16-byte stores.
//   Ghost cells take the wrapped value new(xw, yw), recomputed from the current buffer
//   whose ring is valid, so the written buffer leaves with its ring already exchanged:
//   no second launch.  A generation of a small board is a few latencies long, so a wave
//   issues all its loads before it uses any: a chunk's ghost columns (at most one pair, for
//   W >= 16) take six words loaded with everything else, and chunks of the ghost rows are
//   computed whole, like the others, from the rows they wrap to.  Per generation, against
//   recomputing ghost cells one by one: 100 x 100 5.1 us for 12.7, 1000 x 777 5.0 for 7.9,
//   4096^2 9.9 for 15.7; 8192^2 25.8 for 32.7 (5.2 TB/s: the rate of a copy).
//
// CHOSEN: gol_bits.hip (bit-packed copy of the field, 32 cells per word) from 32 cells a row on,
//   this byte kernel below.
#include "common.hpp"

using namespace appfis;

namespace gol {

__device__ __forceinline__ uint32_t abyte(uint32_t hi, uint32_t lo, uint32_t s)
{
    return __builtin_amdgcn_alignbyte(hi, lo, s);
}

// CB bytes starting `off` bytes (0..15, compile time) into the CB + 16 bytes a[], plus
// the byte before (left) and after (right) that window.
template <int OFF, int CB>
__device__ __forceinline__ void window(const uint32_t (&a)[CB / 4 + 4], uint32_t (&w)[CB / 4], uint32_t& left,
                                       uint32_t& right)
{
    constexpr int D = OFF >> 2, S = OFF & 3;
#pragma unroll
    for (int d = 0; d < CB / 4; d++) {
        if constexpr (S == 0) w[d] = a[D + d];
        else w[d] = abyte(a[D + d + 1], a[D + d], S);
    }
    constexpr int L = OFF - 1, R = OFF + CB;  // byte positions in a[]
    left = (a[L >> 2] >> ((L & 3) * 8)) & 0xFFu;
    right = (a[R >> 2] >> ((R & 3) * 8)) & 0xFFu;
}

// Row of a byte offset p < 2^31 of rows of W >= 2 bytes, by multiply-high: with
// 2^(l-1) < W <= 2^l and m = floor(2^(31+l) / W) + 1 (< 2^32),
// floor(p*m / 2^(31+l)) = floor(p / W), because the excess p*(m - 2^(31+l)/W)/2^(31+l)
// is below 2^31/2^(31+l) <= 1/W.
struct RowDiv {
    uint32_t m;
    int sh;  // l - 1
    __device__ __forceinline__ int row(int p) const { return (int)(__umulhi((uint32_t)p, m) >> sh); }
};

inline RowDiv make_rowdiv(int W)
{
    int l = 0;
    while ((1LL << l) < W) l++;
    RowDiv r;
    r.m = (uint32_t)((1ULL << (31 + l)) / (uint64_t)W + 1ULL);
    r.sh = l - 1;
    return r;
}

__device__ __forceinline__ uint32_t zero_bytes(uint32_t t)
{
    // bytes of t are <= 0x0B: (t + 0x7F) sets bit 7 exactly for non-zero bytes
    return (~(t + 0x7F7F7F7Fu) & 0x80808080u) >> 7;
}

__device__ __forceinline__ uint8_t rule(int n, uint8_t alive) { return (uint8_t)(n == 3 || (n == 2 && alive)); }

// New value of cell (x, y) of the padded buffer, ghost cells mapped to the wrapped
// interior cell; neighbours read from the current buffer (valid ring).
__device__ inline uint8_t cell_new(const uint8_t* __restrict__ u, int W, int H, int x, int y)
{
    const int nx = W - 2, ny = H - 2;
    int xw = x == 0 ? nx : (x == W - 1 ? 1 : x);
    int yw = y == 0 ? ny : (y == H - 1 ? 1 : y);
    const uint8_t* r0 = u + (size_t)(yw - 1) * W;
    const uint8_t* r1 = r0 + W;
    const uint8_t* r2 = r1 + W;
    int n = r0[xw - 1] + r0[xw] + r0[xw + 1] + r1[xw - 1] + r1[xw + 1] + r2[xw - 1] + r2[xw] + r2[xw + 1];
    return rule(n, r1[xw]);
}

// CB cells by SWAR: the rows above, at and below them and the sums of the columns on their
// left and right.  alive' = (n == 3) | (alive & n == 2) = ((n | alive) == 3) for n <= 8.
template <int ND>
__device__ __forceinline__ void next_cells(const uint32_t (&up)[ND], const uint32_t (&m)[ND], const uint32_t (&dn)[ND],
                                           uint32_t sl, uint32_t sr, uint32_t (&out)[ND])
{
    uint32_t s[ND];  // column sums (bytes <= 3), then x-1 / x+1 shifted copies
#pragma unroll
    for (int d = 0; d < ND; d++) s[d] = up[d] + m[d] + dn[d];
#pragma unroll
    for (int d = 0; d < ND; d++) {
        const uint32_t lo = d == 0 ? (sl << 24) : s[d - 1];
        const uint32_t hi = d == ND - 1 ? sr : s[d + 1];
        const uint32_t n = abyte(s[d], lo, 3) + s[d] + abyte(hi, s[d], 1) - m[d];
        out[d] = zero_bytes((n | m[d]) ^ 0x03030303u);
    }
}

// The 3 x 3 cells around one cell: a word from any address of each of three rows W apart, that
// ends with the row's three cells (HIGH) or starts with them.
struct Around {
    uint32_t above, at, below;
};
template <bool HIGH>
__device__ __forceinline__ Around load_around(const uint8_t* __restrict__ u, int first, int W)
{
    const uint8_t* p = u + first - (HIGH ? 1 : 0);
    Around a;
    __builtin_memcpy(&a.above, p, 4);
    __builtin_memcpy(&a.at, p + W, 4);
    __builtin_memcpy(&a.below, p + 2 * W, 4);
    return a;
}
template <bool HIGH>
__device__ __forceinline__ uint32_t next_cell(const Around& a)
{
    constexpr int S = HIGH ? 8 : 0;
    const uint32_t s = (a.above + a.at + a.below) >> S, alive = (a.at >> (8 + S)) & 1u;  // bytes <= 3
    const uint32_t n = (s & 0xFFu) + ((s >> 8) & 0xFFu) + ((s >> 16) & 0xFFu) - alive;
    return (n | alive) == 3u ? 1u : 0u;
}

// Four bytes from any offset, those outside the buffer undefined: the load, from the nearest
// offset inside, and, once it is there, the move of its bytes to their places.
__device__ __forceinline__ uint32_t load_word(const uint8_t* __restrict__ u, int off, int nbytes)
{
    uint32_t x;
    __builtin_memcpy(&x, u + min(max(off, 0), nbytes - 4), 4);
    return x;
}
__device__ __forceinline__ uint32_t place_word(uint32_t x, int off, int nbytes)
{
    const int sh = (off - min(max(off, 0), nbytes - 4)) * 8;
    return sh < 0 ? x << (-sh & 31) : x >> (sh & 31);
}

template <int ND>
__device__ __forceinline__ void set_byte(uint32_t (&w)[ND], int b, uint32_t x)  // b < 0 or >= 4*ND: none
{
#pragma unroll
    for (int d = 0; d < ND; d++) {
        const uint32_t mask = (unsigned)(b - 4 * d) < 4u ? 0xFFu << (((unsigned)b & 3u) * 8) : 0u;
        w[d] = (w[d] & ~mask) | (mask & (x * 0x01010101u));
    }
}

template <int DB, int CB>
__global__ __launch_bounds__(256) void k_gol_plain(const uint8_t* __restrict__ u, uint8_t* __restrict__ v, int W,
                                                   int H, int nchunks, int nbytes, RowDiv rd)
{
    constexpr int ND = CB / 4;   // dwords of a chunk
    constexpr int NA = ND + 4;   // dwords of the aligned span holding a neighbour row's window
    // above-row window starts at p - W: offset (16 - DB) % 16 in its aligned span;
    // below-row window starts at p + W: offset DB.
    constexpr int DA = (16 - DB) & 15;
    // nbytes < 2^31 (checked on the host): 32-bit offsets throughout
    // blocks two apart read each other's rows: keep them on one XCD (shared L2)
    const int c = (int)(xcd_tile(blockIdx.x, gridDim.x) * 256 + threadIdx.x);
    const int lane = threadIdx.x & 63;
    const int p0 = c * CB;
    const bool valid = c < nchunks;
    const bool full = valid && p0 + CB <= nbytes;

    // Rows shorter than a chunk, several of whose boundaries it holds: cell by cell, the loads of
    // four at once (3 x 3000 10.1 -> 8.8 us a generation).  A row of CB bytes is one chunk, whose
    // first and last byte are its ghost cells (14 x 100000 4.5 us, cell by cell 15).
    if (W < CB) {
        if (!valid) return;
#pragma unroll 1
        for (int b = 0; b < CB; b += 4) {
            uint8_t next[4];
#pragma unroll
            for (int k = 0; k < 4; k++) {
                const int p = min(p0 + b + k, nbytes - 1), y = rd.row(p);
                next[k] = cell_new(u, W, H, p - y * W, y);
            }
#pragma unroll
            for (int k = 0; k < 4; k++)
                if (p0 + b + k < nbytes) v[p0 + b + k] = next[k];
        }
        return;
    }
    // rows of the first and last cell of the chunk, and whether the fast path applies
    // (all CB cells in interior rows and every load in bounds) -- before any load, so
    // that all loads of the lane are in flight together
    const int y0 = rd.row(p0);
    const int y1 = rd.row(p0 + CB - 1);
    const int below_end = ((p0 + W) & ~15) + 4 * NA;
    const bool fast = full && y0 >= 1 && y1 <= H - 2 && p0 - W >= 16 && below_end <= nbytes;
    // centre chunk (every valid full lane loads it; shared with neighbours below) and,
    // on the fast path, the aligned spans holding the rows above and below
    uint32_t m[ND], a8[NA], b8[NA];
#pragma unroll
    for (int d = 0; d < ND; d++) m[d] = 0u;
    uint32_t mlb = 0u, mrb = 0u;
    if (full) {
#pragma unroll
        for (int q = 0; q < ND / 4; q++) {
            const uint4 t = *(const uint4*)(u + p0 + 16 * q);
            m[4 * q] = t.x; m[4 * q + 1] = t.y; m[4 * q + 2] = t.z; m[4 * q + 3] = t.w;
        }
    }
    if (fast) {
        const int pa = (p0 - W) & ~15, pb = (p0 + W) & ~15;
#pragma unroll
        for (int q = 0; q < NA / 4; q++) {
            const uint4 ta = *(const uint4*)(u + pa + 16 * q);
            a8[4 * q] = ta.x; a8[4 * q + 1] = ta.y; a8[4 * q + 2] = ta.z; a8[4 * q + 3] = ta.w;
            const uint4 tb = *(const uint4*)(u + pb + 16 * q);
            b8[4 * q] = tb.x; b8[4 * q + 1] = tb.y; b8[4 * q + 2] = tb.z; b8[4 * q + 3] = tb.w;
        }
        // the centre row's outer neighbours for lanes whose adjacent lane does not hold them
        if (lane == 0 || c == 0) mlb = u[p0 - 1];
        if (lane == 63 || c + 1 >= nchunks || p0 + 2 * CB > nbytes) mrb = u[p0 + CB];
    }
    // the chunk's ghost columns: byte br is the right one of row y0, byte bl the left one of the
    // row after it, or of row y0 where the chunk starts with it
    const int nx = W - 2, ny = H - 2;
    auto wrap = [&](int y) { return y == 0 ? ny : (y == H - 1 ? 1 : y); };
    const int x0 = p0 - y0 * W;
    const int br = W - 1 - x0, bl = x0 == 0 ? 0 : br + 1;
    const bool has_r = valid && br < CB && p0 + br < nbytes, has_l = valid && bl < CB && p0 + bl < nbytes;
    // a chunk of a ghost row, at the buffer's ends, or whose aligned spans leave it: the CB
    // cells of row y0, and those of row y0 + 1 if the chunk reaches into it, from the rows
    // they wrap to
    const bool two = br + 1 < CB && p0 + br + 1 < nbytes;
    uint32_t a[2][3][ND + 1];  // from the byte before the chunk's on, three rows of each part
    auto part_at = [&](int part, int k, int d) {
        return p0 - 1 + (wrap(y0 + part) - (y0 + part) + k - 1) * W + 4 * d;
    };
    auto load_part = [&](int part) {
#pragma unroll
        for (int k = 0; k < 3; k++)
#pragma unroll
            for (int d = 0; d <= ND; d++) a[part][k][d] = load_word(u, part_at(part, k, d), nbytes);
    };
    if (valid && !fast) {
        load_part(0);
        if (two) load_part(1);
    }
    Around gr = {}, gl = {};
    if (has_r) gr = load_around<false>(u, (wrap(y0) - 1) * W, W);
    if (has_l) gl = load_around<true>(u, (wrap(x0 == 0 ? y0 : y0 + 1) - 1) * W + nx - 1, W);
    // left / right neighbour bytes of the centre row from the adjacent lanes
    const uint32_t prevl = __shfl_up(m[ND - 1], 1, 64);
    const uint32_t next0 = __shfl_down(m[0], 1, 64);

    if (fast) {
        const uint32_t ml = (lane == 0 || c == 0) ? mlb : (prevl >> 24);
        const uint32_t mr = (lane == 63 || c + 1 >= nchunks || p0 + 2 * CB > nbytes) ? mrb : (next0 & 0xFFu);
        uint32_t up[ND], dn[ND], ul, ur, dl, dr;
        if constexpr (DA == 0) {
            // W multiple of 16: the window is the aligned span's start; edge bytes come
            // from the neighbouring bytes (loaded directly: in bounds by the fast test)
#pragma unroll
            for (int d = 0; d < ND; d++) { up[d] = a8[d]; dn[d] = b8[d]; }
            ul = u[p0 - W - 1];
            ur = a8[ND] & 0xFFu;
            dl = u[p0 + W - 1];
            dr = b8[ND] & 0xFFu;
        } else {
            window<DA, CB>(a8, up, ul, ur);
            window<DB, CB>(b8, dn, dl, dr);
        }
        uint32_t out[ND];
        next_cells(up, m, dn, ul + ml + dl, ur + mr + dr, out);
        if (has_r) set_byte(out, br, next_cell<false>(gr));
        if (has_l) set_byte(out, bl, next_cell<true>(gl));
#pragma unroll
        for (int q = 0; q < ND / 4; q++) {
            uint4 o;
            o.x = out[4 * q]; o.y = out[4 * q + 1]; o.z = out[4 * q + 2]; o.w = out[4 * q + 3];
            *(uint4*)(v + p0 + 16 * q) = o;
        }
    } else if (valid) {
        auto part_cells = [&](int part, uint32_t (&o)[ND]) {
            uint32_t w[3][ND], sl = 0, sr = 0;
#pragma unroll
            for (int k = 0; k < 3; k++) {
                uint32_t x[ND + 1];
#pragma unroll
                for (int d = 0; d <= ND; d++) x[d] = place_word(a[part][k][d], part_at(part, k, d), nbytes);
#pragma unroll
                for (int d = 0; d < ND; d++) w[k][d] = abyte(x[d + 1], x[d], 1);
                sl += x[0] & 0xFFu;
                sr += (x[ND] >> 8) & 0xFFu;
            }
            next_cells(w[0], w[1], w[2], sl, sr, o);
        };
        uint32_t out[ND];
        part_cells(0, out);
        if (two) {
            uint32_t o[ND];
            part_cells(1, o);
#pragma unroll
            for (int d = 0; d < ND; d++) {
                const int keep = min(max(br + 1 - 4 * d, 0), 4);  // bytes up to br are row y0's
                const uint32_t mask = keep == 0 ? 0u : 0xFFFFFFFFu >> (32 - 8 * keep);
                out[d] = (out[d] & mask) | (o[d] & ~mask);
            }
        }
        if (has_r) set_byte(out, br, next_cell<false>(gr));
        if (has_l) set_byte(out, bl, next_cell<true>(gl));
        if (full) {
#pragma unroll
            for (int q = 0; q < ND / 4; q++) {
                uint4 o;
                o.x = out[4 * q]; o.y = out[4 * q + 1]; o.z = out[4 * q + 2]; o.w = out[4 * q + 3];
                *(uint4*)(v + p0 + 16 * q) = o;
            }
        } else {
#pragma unroll
            for (int b = 0; b < CB; b++)
                if (p0 + b < nbytes) v[p0 + b] = (uint8_t)(out[b >> 2] >> ((b & 3) * 8));
        }
    }
}

constexpr int CHUNK = 16;  // bytes (cells) per lane (32 measured slower: fewer lanes in flight)

typedef void (*gol_kernel_t)(const uint8_t*, uint8_t*, int, int, int, int, RowDiv);

}  // namespace gol

// whether the context's workspace holds the packed board, growing it where it can
bool gol_bits_workspace(appfis_ctx* ctx, int nx, int ny);
int gol_bits_run(appfis_ctx* ctx, uint8_t* b0, uint8_t* b1, int nx, int ny, int gens, int force);

extern "C" int appfis_gol(appfis_ctx* ctx, uint8_t* buf0, uint8_t* buf1, int nx, int ny, int gens, int variant,
                          int tsteps)
{
    (void)tsteps;  // reserved: the blocked kernels' depth comes from the tuned candidate
    APPFIS_REQUIRE(ctx && buf0 && buf1, "NULL argument");
    APPFIS_REQUIRE(buf0 != buf1, "the two buffers must differ");
    APPFIS_REQUIRE(nx >= 2 && ny >= 2, "periodic GoL needs an interior of at least 2x2 (got %dx%d)", nx, ny);
    APPFIS_REQUIRE((double)(nx + 2) * (ny + 2) < 2147483647.0, "grid exceeds the int index range");
    APPFIS_REQUIRE(gens >= 0, "gens must be >= 0");
    APPFIS_REQUIRE(((uintptr_t)buf0 & 15) == 0 && ((uintptr_t)buf1 & 15) == 0, "GoL buffers must be 16-byte aligned");
    if (gens == 0) return APPFIS_OK;
    APPFIS_REQUIRE(variant >= 0, "gol: unknown variant %d", variant);
    if (variant >= APPFIS_CANDIDATE0)  // a forced blocked candidate of the bit-packed form
        return gol_bits_run(ctx, buf0, buf1, nx, ny, gens, variant - APPFIS_CANDIDATE0);
    // the bit-packed form needs a word of cells; narrower boards run the byte kernel, which
    // gives the same bytes, and so do boards whose width is no multiple of 32 where there is
    // no workspace (a first call while the stream is being captured)
    if (variant == APPFIS_CHOSEN && nx >= 32 && (nx % 32 == 0 || gol_bits_workspace(ctx, nx, ny)))
        return gol_bits_run(ctx, buf0, buf1, nx, ny, gens, -1);
    const int W = nx + 2, H = ny + 2;
    const int nbytes = W * H;
    const int nchunks = (nbytes + gol::CHUNK - 1) / gol::CHUNK;
    static constexpr gol::gol_kernel_t table[16] = {
        gol::k_gol_plain<0, gol::CHUNK>,  gol::k_gol_plain<1, gol::CHUNK>,  gol::k_gol_plain<2, gol::CHUNK>,
        gol::k_gol_plain<3, gol::CHUNK>,  gol::k_gol_plain<4, gol::CHUNK>,  gol::k_gol_plain<5, gol::CHUNK>,
        gol::k_gol_plain<6, gol::CHUNK>,  gol::k_gol_plain<7, gol::CHUNK>,  gol::k_gol_plain<8, gol::CHUNK>,
        gol::k_gol_plain<9, gol::CHUNK>,  gol::k_gol_plain<10, gol::CHUNK>, gol::k_gol_plain<11, gol::CHUNK>,
        gol::k_gol_plain<12, gol::CHUNK>, gol::k_gol_plain<13, gol::CHUNK>, gol::k_gol_plain<14, gol::CHUNK>,
        gol::k_gol_plain<15, gol::CHUNK>};
    gol::gol_kernel_t k = table[W & 15];
    // the ring of the input buffer must be valid (reference: ExchangeInitial on both
    // buffers in InitializeExecution, Runtime.hpp:124-142)
    const int dims[2] = {W, H};
    int st = appfis_exchange(ctx, buf0, APPFIS_U8, 2, dims, 1, 1);
    if (st) return st;
    uint8_t* buf[2] = {buf0, buf1};
    const unsigned blocks = ceil_div((size_t)nchunks, 256);
    const gol::RowDiv rd = gol::make_rowdiv(W);
    st = ktime_begin(ctx);
    if (st) return st;
    for (int g = 0; g < gens; g++) {
        hipLaunchKernelGGL(k, dim3(blocks), dim3(256), 0, ctx->stream, buf[g & 1], buf[(g + 1) & 1], W, H, nchunks,
                           nbytes, rd);
        APPFIS_LAUNCH_CHECK();
    }
    return ktime_end(ctx, gens, gens);
}
