// GameOfLife CHOSEN form: the same B3/S23 generations on a bit-packed copy of the field.
//
// The call packs the interior of the uint8 field into 32-bit words (bit b of word w of
// row y = cell (32w + b, y), interior coordinates), advances the packed field (many
// generations per launch), and its last launch computes the last generation while
// unpacking the last two back into the two uint8 buffers, rings exchanged: on return both
// buffers hold exactly what the PLAIN form leaves (generation `gens` in buf[gens % 2],
// generation gens-1 in the other).  A row takes ceil(nx / 32) words; where nx is no multiple
// of 32 the rest of its last word means nothing, and the kernels join the row's end and start
// by shifting.  Cells must hold 0 or 1.
//
// One generation, per word, with 32 cells evaluated at once by bitwise full adders:
//   h(row)  = W + C + E                (2-bit horizontal sum of each row; W/E are the
//                                       word shifted by one cell, funnel-shifted in from
//                                       the neighbouring words, wrapping at the row end)
//   S       = h(y-1) + h(y) + h(y+1)   (3x3 sum including the cell itself, 0..9)
//   alive'  = (S == 3) | (alive & S == 4)
// A thread owns one word column over K consecutive rows, so each row's horizontal sum
// is computed once and used by the three output rows that need it.
#include "common.hpp"

#include <algorithm>
#include <cmath>

using namespace appfis;

namespace golbits {

// 3-input bitwise functions, one v_bitop3_b32 each (gfx950).  Both are symmetric in
// their inputs, so the lookup table does not depend on the operand order.  Written as
// separate instructions on purpose: sharing a ^ b between the two lets the compiler
// fall back to two-input operations.
__device__ __forceinline__ uint32_t xor3(uint32_t a, uint32_t b, uint32_t c)
{
    return __builtin_amdgcn_bitop3_b32(a, b, c, 0x96);  // a ^ b ^ c
}
__device__ __forceinline__ uint32_t maj(uint32_t a, uint32_t b, uint32_t c)
{
    return __builtin_amdgcn_bitop3_b32(a, b, c, 0xE8);  // at least two of a, b, c
}

// B3/S23 from the adders of the three rows' 2-bit horizontal sums: with s0 = xor3 and
// c0 = maj of the low bit-planes and v1 = xor3, c1 = maj of the high ones, the 3x3 sum
// is S = s0 + 2(c0 + v1) + 4c1, so
//   S == 3  <=>  s0 & P,   P = (c0 ^ v1) & ~c1
//   S == 4  <=>  ~s0 & Q,  Q = ~(c0 ^ v1) & (c0 ^ c1)
// and alive' = (s0 & P) | (alive & ~s0 & Q): four three-input operations (truth-table
// index a*4 + b*2 + c for bitop3(a, b, c)), checked against S == 3 | (alive & S == 4)
// for every triple of 2-bit sums.
__device__ __forceinline__ uint32_t life_rule(uint32_t s0, uint32_t c0, uint32_t v1, uint32_t c1, uint32_t alive)
{
    const uint32_t p = __builtin_amdgcn_bitop3_b32(c0, v1, c1, 0x14);
    const uint32_t q = __builtin_amdgcn_bitop3_b32(c0, v1, c1, 0x42);
    const uint32_t t = __builtin_amdgcn_bitop3_b32(alive, s0, q, 0x20);
    return __builtin_amdgcn_bitop3_b32(s0, p, t, 0xEA);
}

// cells x = 32w .. 32w+31 of interior row y (uint8, 0/1) -> one word
__global__ __launch_bounds__(256) void k_pack(const uint8_t* __restrict__ u, uint32_t* __restrict__ P, int nx,
                                              int ny, int NW)
{
    const size_t t = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (t >= (size_t)NW * ny) return;
    const int y = (int)(t / NW), w = (int)(t - (size_t)y * NW);
    const uint8_t* row = u + (size_t)(y + 1) * (nx + 2) + 1 + 32 * w;
    uint32_t word = 0;
#pragma unroll
    for (int k = 0; k < 8; k++) {
        const uint32_t x = ((uint32_t)row[4 * k] | ((uint32_t)row[4 * k + 1] << 8) |
                            ((uint32_t)row[4 * k + 2] << 16) | ((uint32_t)row[4 * k + 3] << 24)) &
                           0x01010101u;
        // byte j of x (0/1) lands on bit 24 + j: the other partial products fall on
        // distinct bits below 24 or above 31, so nothing carries into bits 24..27
        word |= ((x * 0x01020408u) >> 24) << (4 * k);
    }
    P[t] = word;
}

// One generation of a board whose rows are whole words, K rows of a word column a thread.  Where
// it beats the blocked forms is step_cost's business (see gol_bits_run): calls of two generations,
// and tall boards of few words, in whose windows most lanes hold nothing.
template <int K>
__global__ __launch_bounds__(256) void k_step(const uint32_t* __restrict__ P, uint32_t* __restrict__ Q, int NW, int ny,
                                              unsigned nitems)
{
    // consecutive blocks share rows at their band edges: keep them on one XCD
    const unsigned t = xcd_tile(blockIdx.x, gridDim.x) * 256 + threadIdx.x;
    if (t >= nitems) return;
    const int band = (int)(t / (unsigned)NW), w = (int)(t - (unsigned)band * NW);
    const int wl = w == 0 ? NW - 1 : w - 1;
    const int wr = w == NW - 1 ? 0 : w + 1;
    const int y0 = band * K;
    uint32_t h0[K + 2], h1[K + 2], cen[K + 2];
#pragma unroll
    for (int r = 0; r < K + 2; r++) {
        int y = y0 - 1 + r;  // periodic rows; y < ny + K, so the loop ends (once if K <= ny)
        if (y < 0) y += ny;
        while (y >= ny) y -= ny;
        const uint32_t* row = P + (size_t)y * NW;
        const uint32_t c = row[w], l = row[wl], rr = row[wr];
        const uint32_t W = __builtin_amdgcn_alignbit(c, l, 31);  // cell x-1 at bit x
        const uint32_t E = __builtin_amdgcn_alignbit(rr, c, 1);  // cell x+1 at bit x
        h0[r] = xor3(W, c, E);
        h1[r] = maj(W, c, E);
        cen[r] = c;
    }
#pragma unroll
    for (int k = 0; k < K; k++) {
        const int y = y0 + k;
        if (y >= ny) break;
        // S = h[k] + h[k+1] + h[k+2] through the carry-save adders of the two bit-planes
        const uint32_t s0 = xor3(h0[k], h0[k + 1], h0[k + 2]);
        const uint32_t c0 = maj(h0[k], h0[k + 1], h0[k + 2]);
        const uint32_t u1 = xor3(h1[k], h1[k + 1], h1[k + 2]);
        const uint32_t c1 = maj(h1[k], h1[k + 1], h1[k + 2]);
        Q[(size_t)y * NW + w] = life_rule(s0, c0, u1, c1, cen[k + 1]);
    }
}

constexpr int KROWS = 8;

// 32 cells from cell x on of one padded uint8 row (bit b of word = cell x + b), and the ring
// cells that the periodic exchange (X first) copies from the row: ghost column nx+1 holds
// cell 0, ghost column 0 holds cell nx-1.
__device__ __forceinline__ void put_word(uint8_t* __restrict__ u, size_t W, int prow, int x, bool first, bool last,
                                         uint32_t word)
{
    uint8_t* row = u + (size_t)prow * W;
#pragma unroll
    for (int b = 0; b < 32; b++) row[1 + x + b] = (uint8_t)((word >> b) & 1u);
    if (first) row[W - 1] = (uint8_t)(word & 1u);
    if (last) row[0] = (uint8_t)(word >> 31);
}

// The last generation of a call fused with the unpacking: from the packed generation
// n-1 in P it computes generation n and writes generation n into `un`
// and generation n-1 into `uprev`, both with their periodic rings -- what one generation,
// unpacking both generations and exchanging both rings would leave, in one pass.  Where nx is
// no multiple of 32 the thread of the last word takes the row's last 32 cells, which overlap
// the word before it (both write the same bytes there), so that every thread moves whole
// words.  The exchange's Y step copies
// padded row ny (ghost columns included) into ghost row 0 and padded row 1 into ghost
// row ny+1, so the thread of interior row ny-1 also writes row 0 and that of row 0 also
// writes row ny+1.  Reads only P: `uprev` may be the buffer the call's input came from.
template <int K>
__global__ __launch_bounds__(256) void k_step_unpack(const uint32_t* __restrict__ P, uint8_t* __restrict__ un,
                                                     uint8_t* __restrict__ uprev, int nx, int NW, int ny,
                                                     unsigned nitems)
{
    const unsigned t = xcd_tile(blockIdx.x, gridDim.x) * 256 + threadIdx.x;
    if (t >= nitems) return;
    const int band = (int)(t / (unsigned)NW), w = (int)(t - (unsigned)band * NW);
    const int wl = w == 0 ? NW - 1 : w - 1;
    const int wr = w == NW - 1 ? 0 : w + 1;
    const int y0 = band * K;
    const size_t W = (size_t)nx + 2;
    const unsigned rem = (unsigned)nx & 31u;  // cells of the last word, 0: all 32
    const bool first = w == 0, last = w == NW - 1, end = last && rem != 0;
    const int x = end ? nx - 32 : 32 * w;     // first cell of this thread's 32
    uint32_t h0[K + 2], h1[K + 2], cen[K + 2];
#pragma unroll
    for (int r = 0; r < K + 2; r++) {
        int y = y0 - 1 + r;  // periodic rows; y < ny + K, so the loop ends (once if K <= ny)
        if (y < 0) y += ny;
        while (y >= ny) y -= ny;
        const uint32_t* row = P + (size_t)y * NW;
        const uint32_t cw = row[w], lw = row[wl], rr = row[wr];
        const uint32_t c = end ? __builtin_amdgcn_alignbit(cw, lw, rem) : cw;
        // bit 31 of l is the cell left of the 32: cell nx-1 for the first word, and the last
        // cell but 32 of a row whose last word is not full
        const uint32_t l = (first || end) && rem != 0 ? lw << (32u - rem) : lw;
        const uint32_t Wc = __builtin_amdgcn_alignbit(c, l, 31);   // cell x-1 at bit x
        const uint32_t Ec = __builtin_amdgcn_alignbit(rr, c, 1);   // cell x+1 at bit x
        h0[r] = xor3(Wc, c, Ec);
        h1[r] = maj(Wc, c, Ec);
        cen[r] = c;
    }
#pragma unroll
    for (int k = 0; k < K; k++) {
        const int y = y0 + k;
        if (y >= ny) break;
        const uint32_t s0 = xor3(h0[k], h0[k + 1], h0[k + 2]);
        const uint32_t c0 = maj(h0[k], h0[k + 1], h0[k + 2]);
        const uint32_t u1 = xor3(h1[k], h1[k + 1], h1[k + 2]);
        const uint32_t c1 = maj(h1[k], h1[k + 1], h1[k + 2]);
        const uint32_t next = life_rule(s0, c0, u1, c1, cen[k + 1]);
        put_word(un, W, y + 1, x, first, last, next);
        put_word(uprev, W, y + 1, x, first, last, cen[k + 1]);
        if (y == ny - 1) {
            put_word(un, W, 0, x, first, last, next);
            put_word(uprev, W, 0, x, first, last, cen[k + 1]);
        }
        if (y == 0) {
            put_word(un, W, ny + 1, x, first, last, next);
            put_word(uprev, W, ny + 1, x, first, last, cen[k + 1]);
        }
    }
}

// Temporal blocking: G generations per launch.  A block of NWAVES waves spans whole
// packed rows: NW = 64*WX words, lane l of wave (wx, wy) owns word 64*wx + l, and wave
// row wy holds K consecutive rows in registers, so the block's window is WY*K rows of
// the full periodic row width.  Its centre OUT = WY*K - 2G rows are exact after G
// generations (each generation invalidates one more window row at each end); blocks
// are spaced OUT rows apart.  Per generation:
//   A  each wave publishes its lane-0 and lane-63 words (all K rows) to LDS; barrier
//   B  horizontal sums of its K rows: the neighbour words come from lanes l-1 / l+1 by
//      DPP wave shifts, and across wave edges (lanes 0 / 63) from the LDS words of the
//      waves left / right (periodic in wx); the first and last rows' sums go to LDS;
//      barrier
//   C  vertical combine: the sums of the rows above / below the wave's band come from
//      the waves above / below (zero outside the window), then the rule.
// Never chosen any more (48 generations at 16384 x 16384: 441 us, windows 171; at 2048 x 2048
// 107, windows 24); kept as a forced candidate, the form that spreads a row over waves.
template <int K, int G, int NWAVES>
__global__ __launch_bounds__(64 * NWAVES) void k_step_tb(const uint32_t* __restrict__ P, uint32_t* __restrict__ Q,
                                                          int NW, int ny, int WX, int OUT, int gens)
{
    __shared__ uint32_t edge_lo[NWAVES][K], edge_hi[NWAVES][K];  // lane-0 / lane-63 words
    __shared__ uint32_t sum_top[2][NWAVES][64], sum_bot[2][NWAVES][64];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int wx = wv % WX, wy = wv / WX;
    const int WY = NWAVES / WX;
    const int w = wx * 64 + lane;
    const int left = wy * WX + (wx == 0 ? WX - 1 : wx - 1);
    const int right = wy * WX + (wx == WX - 1 ? 0 : wx + 1);
    // bands in XCD-contiguous order: neighbouring bands (whose rows form each other's halo)
    // run on one XCD and share its L2
    const int band = (int)xcd_tile(blockIdx.x, gridDim.x);
    const int y0 = band * OUT - G + wy * K;  // global row of register row 0
    // periodic row of register row 0 (the window may start up to G rows below 0 and end
    // past ny); then consecutive rows step by one word row, wrapping once at ny when
    // K <= ny (the general loop otherwise).  32-bit word offsets: NW * ny < 2^31.
    int yw = y0 % ny;
    if (yw < 0) yw += ny;
    uint32_t R[K];
    if (K <= ny) {
        int y = yw, off = yw * NW + w;
#pragma unroll
        for (int k = 0; k < K; k++) {
            R[k] = P[off];
            ++y;
            off += NW;
            if (y == ny) {
                y = 0;
                off = w;
            }
        }
    } else {
#pragma unroll
        for (int k = 0; k < K; k++) {
            int y = yw + k;
            while (y >= ny) y -= ny;
            R[k] = P[y * NW + w];
        }
    }
    for (int g = 0; g < gens; g++) {
        if (lane == 0)
#pragma unroll
            for (int k = 0; k < K; k++) edge_lo[wv][k] = R[k];
        if (lane == 63)
#pragma unroll
            for (int k = 0; k < K; k++) edge_hi[wv][k] = R[k];
        __syncthreads();
        // the neighbouring waves' edge words, read by every lane (one address per wave:
        // LDS broadcast) so that no read waits behind a lane mask
        uint32_t eh[K], el[K];
#pragma unroll
        for (int k = 0; k < K; k++) {
            eh[k] = edge_hi[left][k];
            el[k] = edge_lo[right][k];
        }
        uint32_t h0[K], h1[K];
#pragma unroll
        for (int k = 0; k < K; k++) {
            // lane l receives lane l-1 (wave_shr:1) / lane l+1 (wave_shl:1); lanes 0 / 63
            // have no source lane and keep the `old` operand: the neighbouring wave's word
            const uint32_t l = (uint32_t)__builtin_amdgcn_update_dpp((int)eh[k], (int)R[k], 0x138, 0xF, 0xF, false);
            const uint32_t r = (uint32_t)__builtin_amdgcn_update_dpp((int)el[k], (int)R[k], 0x130, 0xF, 0xF, false);
            const uint32_t c = R[k];
            const uint32_t Wc = __builtin_amdgcn_alignbit(c, l, 31);
            const uint32_t Ec = __builtin_amdgcn_alignbit(r, c, 1);
            h0[k] = xor3(Wc, c, Ec);
            h1[k] = maj(Wc, c, Ec);
        }
        sum_top[0][wv][lane] = h0[0];
        sum_top[1][wv][lane] = h1[0];
        sum_bot[0][wv][lane] = h0[K - 1];
        sum_bot[1][wv][lane] = h1[K - 1];
        __syncthreads();
        uint32_t a0 = 0u, a1 = 0u, z0 = 0u, z1 = 0u;
        if (wy > 0) {
            a0 = sum_bot[0][wv - WX][lane];
            a1 = sum_bot[1][wv - WX][lane];
        }
        if (wy < WY - 1) {
            z0 = sum_top[0][wv + WX][lane];
            z1 = sum_top[1][wv + WX][lane];
        }
#pragma unroll
        for (int k = 0; k < K; k++) {
            const uint32_t u0 = k == 0 ? a0 : h0[k - 1], u1 = k == 0 ? a1 : h1[k - 1];
            const uint32_t d0 = k == K - 1 ? z0 : h0[k + 1], d1 = k == K - 1 ? z1 : h1[k + 1];
            const uint32_t s0 = xor3(u0, h0[k], d0);
            const uint32_t c0 = maj(u0, h0[k], d0);
            const uint32_t v1 = xor3(u1, h1[k], d1);
            const uint32_t c1 = maj(u1, h1[k], d1);
            R[k] = life_rule(s0, c0, v1, c1, R[k]);
        }
    }
    // output rows: window rows G .. G+OUT-1 of the block, global rows band*OUT + r
    const int ybase = band * OUT - G + wy * K;
#pragma unroll
    for (int k = 0; k < K; k++) {
        const int r = wy * K + k - G;  // output row within the block's OUT rows
        const int y = ybase + k;
        if (r >= 0 && r < OUT && y < ny) Q[y * NW + w] = R[k];
    }
}

// Full-row waves: each wave holds K rows of the whole packed width, NW = 64 * WPL words,
// lane l holding words WPL*l .. WPL*l + WPL - 1 of each row.  A word's horizontal
// neighbours are then the lane's own registers, except at the lane's two ends, which
// come from the adjacent lanes by DPP wave rotates (wave_ror / wave_rol), and the
// rotation is the periodic wrap of the row: no LDS for the horizontal direction, and
// 16-byte loads and stores.  The block's NWAVES waves stack bands of K rows.  Each
// generation a wave publishes the horizontal sums (both bit-planes) of its first and
// last rows into LDS slots double-buffered by generation parity; after the one barrier
// it reads the sums of the rows just above and below its band (zero outside the
// block's window).  A wave still reading generation g's slots is never overwritten:
// the next writes to them come after the barrier of generation g+1, which every wave
// reaches only after finishing g.  G generations per launch, OUT = NWAVES*K - 2G
// output rows per block.  Window row r holds a valid state after generation g (counted
// from 0) only for g + 1 <= r <= NWAVES*K - 2 - g: the waves at the window's ends skip
// the rule once all their rows are past that range, and their horizontal sums once
// their rows were already past it before the generation (nothing valid reads them then;
// they still meet every barrier).
template <int WPL>
struct WordVec;
template <> struct WordVec<1> {
    using V = uint32_t;
    __device__ static void get(const V& v, uint32_t (&w)[1]) { w[0] = v; }
    __device__ static V put(const uint32_t (&w)[1]) { return w[0]; }
};
template <> struct WordVec<2> {
    using V = uint2;
    __device__ static void get(const V& v, uint32_t (&w)[2]) { w[0] = v.x; w[1] = v.y; }
    __device__ static V put(const uint32_t (&w)[2]) { return make_uint2(w[0], w[1]); }
};
template <> struct WordVec<4> {
    using V = uint4;
    __device__ static void get(const V& v, uint32_t (&w)[4]) { w[0] = v.x; w[1] = v.y; w[2] = v.z; w[3] = v.w; }
    __device__ static V put(const uint32_t (&w)[4]) { return make_uint4(w[0], w[1], w[2], w[3]); }
};

// The generation loop of the full-row form: `gens` generations of the K rows in R
// (window rows wv*K .. wv*K+K-1 of the block); with KEEP, Rp receives the rows as they
// were before the last generation.
template <int WPL, int K, int G, int NWAVES, bool KEEP>
__device__ __forceinline__ void tw_generations(uint32_t (&R)[K][WPL], uint32_t (&Rp)[K][WPL],
                                               uint32_t (*hs)[NWAVES][2][2][64 * WPL], int lane, int wv, int gens)
{
    using VW = WordVec<WPL>;
    using V = typename VW::V;
    const int top = wv * K, bot = wv * K + K - 1, last = NWAVES * K - 1;  // window rows of the wave
    for (int g = 0; g < gens; g++) {
        const int b = g & 1;
        const bool sums = bot >= g && top <= last - g;        // some row valid before generation g
        const bool rule = bot >= g + 1 && top <= last - 1 - g;  // some row valid after it
        if constexpr (KEEP) {
            if (g == gens - 1) {
#pragma unroll
                for (int k = 0; k < K; k++)
#pragma unroll
                    for (int w = 0; w < WPL; w++) Rp[k][w] = R[k][w];
            }
        }
        uint32_t h0[K + 2][WPL], h1[K + 2][WPL];
        if (sums) {
#pragma unroll
            for (int k = 0; k < K; k++) {
                // the words left of the lane's first and right of its last (periodic row;
                // a rotation has a source for every lane)
                const uint32_t lft = (uint32_t)__builtin_amdgcn_mov_dpp((int)R[k][WPL - 1], 0x13C, 0xF, 0xF, true);
                const uint32_t rgt = (uint32_t)__builtin_amdgcn_mov_dpp((int)R[k][0], 0x134, 0xF, 0xF, true);
#pragma unroll
                for (int w = 0; w < WPL; w++) {
                    const uint32_t c = R[k][w];
                    const uint32_t l = w == 0 ? lft : R[k][w - 1];
                    const uint32_t r = w == WPL - 1 ? rgt : R[k][w + 1];
                    const uint32_t Wc = __builtin_amdgcn_alignbit(c, l, 31);
                    const uint32_t Ec = __builtin_amdgcn_alignbit(r, c, 1);
                    h0[k + 1][w] = xor3(Wc, c, Ec);
                    h1[k + 1][w] = maj(Wc, c, Ec);
                }
            }
            reinterpret_cast<V*>(hs[b][wv][0][0])[lane] = VW::put(h0[1]);
            reinterpret_cast<V*>(hs[b][wv][0][1])[lane] = VW::put(h1[1]);
            reinterpret_cast<V*>(hs[b][wv][1][0])[lane] = VW::put(h0[K]);
            reinterpret_cast<V*>(hs[b][wv][1][1])[lane] = VW::put(h1[K]);
        }
        __syncthreads();
        if (!rule) continue;
        {
            // rows -1 and K: whole-vector reads from the neighbouring waves' slots.  The
            // block's first and last waves read their own slots instead: rows outside the
            // window only reach the halo rows, which are never stored.
            const int up = wv > 0 ? wv - 1 : wv, dn = wv < NWAVES - 1 ? wv + 1 : wv;
            VW::get(reinterpret_cast<const V*>(hs[b][up][1][0])[lane], h0[0]);
            VW::get(reinterpret_cast<const V*>(hs[b][up][1][1])[lane], h1[0]);
            VW::get(reinterpret_cast<const V*>(hs[b][dn][0][0])[lane], h0[K + 1]);
            VW::get(reinterpret_cast<const V*>(hs[b][dn][0][1])[lane], h1[K + 1]);
        }
#pragma unroll
        for (int k = 0; k < K; k++)
#pragma unroll
            for (int w = 0; w < WPL; w++) {
                const uint32_t s0 = xor3(h0[k][w], h0[k + 1][w], h0[k + 2][w]);
                const uint32_t c0 = maj(h0[k][w], h0[k + 1][w], h0[k + 2][w]);
                const uint32_t v1 = xor3(h1[k][w], h1[k + 1][w], h1[k + 2][w]);
                const uint32_t c1 = maj(h1[k][w], h1[k + 1][w], h1[k + 2][w]);
                R[k][w] = life_rule(s0, c0, v1, c1, R[k][w]);
            }
    }
}

template <int WPL, int K, int G, int NWAVES>
__global__ __launch_bounds__(64 * NWAVES) void k_step_tw(const uint32_t* __restrict__ P, uint32_t* __restrict__ Q,
                                                          int NW, int ny, int OUT, int gens)
{
    using VW = WordVec<WPL>;
    using V = typename VW::V;
    // [parity][wave][first / last row][bit-plane][word of the row]
    __shared__ uint32_t hs[2][NWAVES][2][2][64 * WPL];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int band = (int)xcd_tile(blockIdx.x, gridDim.x);  // XCD-contiguous band order
    const int y0 = band * OUT - G + wv * K;  // global row of register row 0
    int yw = y0 % ny;
    if (yw < 0) yw += ny;
    uint32_t R[K][WPL], Rp[K][WPL];
#pragma unroll
    for (int k = 0; k < K; k++) {
        int y = yw + k;  // periodic rows (the window may wrap more than once when ny < K)
        while (y >= ny) y -= ny;
        VW::get(reinterpret_cast<const V*>(P + (size_t)y * NW)[lane], R[k]);
    }
    tw_generations<WPL, K, G, NWAVES, false>(R, Rp, hs, lane, wv, gens);
    // output rows: window rows G .. G+OUT-1 of the block, global rows band*OUT + r
    const int ybase = band * OUT - G + wv * K;
#pragma unroll
    for (int k = 0; k < K; k++) {
        const int r = wv * K + k - G;
        const int y = ybase + k;
        if (r >= 0 && r < OUT && y < ny) reinterpret_cast<V*>(Q + (size_t)y * NW)[lane] = VW::put(R[k]);
    }
}

// 16 cells of a padded uint8 row from 16 bits (bit j = cell j), as one 16-byte store
// (the compiler merges the byte stores), plus the ghost cell the periodic exchange
// copies from it: chunk 0 holds cell 0, which ghost column nx+1 takes; the last chunk
// holds cell nx-1, which ghost column 0 takes.
// 16 bytes at any address, allowed to alias the uint8 field it reads and writes
typedef unsigned int u32x4_u __attribute__((ext_vector_type(4), aligned(1), may_alias));
__device__ __forceinline__ void put_chunk(uint8_t* __restrict__ row, size_t W, int c, int nchunks, uint32_t h)
{
    u32x4_u d;
#pragma unroll
    for (int q = 0; q < 4; q++) d[q] = (((h >> (4 * q)) & 0xFu) * 0x00204081u) & 0x01010101u;  // bit j -> byte j
    *reinterpret_cast<u32x4_u*>(row + 1 + 16 * c) = d;
    if (c == 0) row[W - 1] = (uint8_t)(h & 1u);
    if (c == nchunks - 1) row[0] = (uint8_t)((h >> 15) & 1u);
}

// The first and last launches of a call, fused with the uint8 conversions of k_pack and
// k_step_unpack.  IN_U8: the window comes from the padded uint8 field u (interior cells
// (x, y) at (y+1)*(nx+2) + 1 + x, 0 or 1) and is packed in registers; else from P.
// OUT_U8: the output rows go out as uint8 -- generation n (the launch's last) into un,
// generation n-1 into uprev, with the periodic ring as the exchange leaves it (the
// block holding interior row ny-1 also writes ghost row 0, the one holding row 0 ghost
// row ny+1) -- else into Q, packed.  The uint8 rows move in 16-byte chunks, chunk
// 64p + l of a row by lane l in pass p, so that each access instruction covers 1 KB of
// the row; the chunks' 16-bit halves of the lanes' words pass through a per-wave row in
// LDS (each lane owns WPL consecutive words).  A launch that reads u must not write it:
// the host pairs IN_U8 and OUT_U8 only across two launches.
template <int WPL, int K, int G, int NWAVES, bool IN_U8, bool OUT_U8>
__global__ __launch_bounds__(64 * NWAVES) void k_step_tw_io(const uint8_t* __restrict__ u, const uint32_t* __restrict__ P,
                                                             uint32_t* __restrict__ Q, uint8_t* __restrict__ un,
                                                             uint8_t* __restrict__ uprev, int nx, int ny, int OUT,
                                                             int gens)
{
    using VW = WordVec<WPL>;
    using V = typename VW::V;
    constexpr int NW = 64 * WPL;  // words of a row
    constexpr int NC = 2 * NW;    // 16-cell chunks of a row
    const size_t W = (size_t)nx + 2;
    __shared__ uint32_t hs[2][NWAVES][2][2][NW];
    __shared__ uint32_t stage[NWAVES][NW];  // one row of the wave, as words
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    // chunk c = half c of the row (little-endian); may_alias: the same LDS is also read
    // and written as words
    typedef uint16_t __attribute__((may_alias)) half_t;
    half_t* st16 = reinterpret_cast<half_t*>(stage[wv]);
    const int band = (int)xcd_tile(blockIdx.x, gridDim.x);
    const int y0 = band * OUT - G + wv * K;
    int yw = y0 % ny;
    if (yw < 0) yw += ny;
    uint32_t R[K][WPL], Rp[K][WPL];
#pragma unroll
    for (int k = 0; k < K; k++) {
        int y = yw + k;
        while (y >= ny) y -= ny;
        if constexpr (IN_U8) {
            const uint8_t* row = u + (size_t)(y + 1) * W + 1;
#pragma unroll
            for (int p = 0; p < NC / 64; p++) {
                const int c = 64 * p + lane;
                const u32x4_u b = *reinterpret_cast<const u32x4_u*>(row + 16 * c);
                uint32_t h = 0;
#pragma unroll
                for (int q = 0; q < 4; q++)
                    h |= (((b[q] & 0x01010101u) * 0x01020408u) >> 24) << (4 * q);  // byte j -> bit j, as in k_pack
                st16[c] = (uint16_t)h;
            }
#pragma unroll
            for (int w = 0; w < WPL; w++) R[k][w] = stage[wv][WPL * lane + w];
        } else {
            VW::get(reinterpret_cast<const V*>(P + (size_t)y * NW)[lane], R[k]);
        }
    }
    tw_generations<WPL, K, G, NWAVES, OUT_U8>(R, Rp, hs, lane, wv, gens);
    const int ybase = band * OUT - G + wv * K;
#pragma unroll
    for (int k = 0; k < K; k++) {
        const int r = wv * K + k - G;
        const int y = ybase + k;
        if (r < 0 || r >= OUT || y >= ny) continue;
        if constexpr (OUT_U8) {
#pragma unroll
            for (int f = 0; f < 2; f++) {
                uint8_t* const dst = f == 0 ? un : uprev;
#pragma unroll
                for (int w = 0; w < WPL; w++) stage[wv][WPL * lane + w] = f == 0 ? R[k][w] : Rp[k][w];
#pragma unroll
                for (int p = 0; p < NC / 64; p++) {
                    const int c = 64 * p + lane;
                    const uint32_t h = st16[c];
                    put_chunk(dst + (size_t)(y + 1) * W, W, c, NC, h);
                    if (y == ny - 1) put_chunk(dst, W, c, NC, h);
                    if (y == 0) put_chunk(dst + (size_t)(ny + 1) * W, W, c, NC, h);
                }
            }
        } else {
            reinterpret_cast<V*>(Q + (size_t)y * NW)[lane] = VW::put(R[k]);
        }
    }
}

// The blocked form for rows of any width nx >= 32 (NW = ceil(nx / 32) words; bits past cell
// nx-1 of a row's last word mean nothing).  A wave's K rows span a window of 64*WPL words of
// which all but the first and the last are stored: G <= 32 generations spoil at most the 32
// cells of a word at either end, so the wrap of tw_generations' rotation does no harm.  Tile
// (tx, band) stores words tx*(64*WPL - 2) .. and OUT = NWAVES*K - 2G rows.  The window is
// periodic in cells, not in words: window word g holds cells 32g .. 32g+31 modulo nx, so where
// the row's end falls inside a word the fetch joins the cells before it and those from cell 0.
template <int WPL, int K, int G, int NWAVES>
__global__ __launch_bounds__(64 * NWAVES) void k_step_win(const uint32_t* __restrict__ P, uint32_t* __restrict__ Q,
                                                          int nx, int NW, int ny, int tiles_x, int gens)
{
    constexpr int OUTW = 64 * WPL - 2, OUT = NWAVES * K - 2 * G;
    static_assert(G <= 32 && OUT > 0, "a halo of one word and of G rows");
    __shared__ uint32_t hs[2][NWAVES][2][2][64 * WPL];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int t = (int)xcd_tile(blockIdx.x, gridDim.x);  // x fastest: neighbouring tiles share an L2
    const int band = t / tiles_x, tx = t - band * tiles_x;
    const int g0 = tx * OUTW - 1 + WPL * lane;  // word of R[.][0]
    int yw = (band * OUT - G + wv * K) % ny;
    if (yw < 0) yw += ny;
    uint32_t R[K][WPL], Rp[K][WPL];
    const bool whole = tx > 0 && 32LL * (tx * OUTW + OUTW + 1) <= nx;  // every word a stored one, and full
    if (whole) {
#pragma unroll
        for (int k = 0; k < K; k++) {
            int y = yw + k;  // periodic rows (the window may wrap more than once when ny < K)
            while (y >= ny) y -= ny;
            const uint32_t* row = P + (size_t)y * NW;
#pragma unroll
            for (int w = 0; w < WPL; w++) R[k][w] = row[g0 + w];
        }
    } else {
        // word g: cells s .. of the row (s = 32g modulo nx) down from bit s & 31 of word ia, `low`
        // of them before the row's end, then cells from 0 on.  Words past the one right of the
        // row's last are not used and hold its first.
        int ia[WPL], ib[WPL];
        unsigned sh[WPL], low[WPL];
#pragma unroll
        for (int w = 0; w < WPL; w++) {
            const int g = g0 + w;
            int sc = g < 0 ? nx - 32 : g > NW ? 0 : 32 * g;
            if (sc >= nx) sc -= nx;
            ia[w] = sc >> 5;
            ib[w] = ia[w] + 1 < NW ? ia[w] + 1 : ia[w];
            sh[w] = (unsigned)sc & 31u;
            low[w] = (unsigned)(nx - sc < 32 ? nx - sc : 32);
        }
#pragma unroll
        for (int k = 0; k < K; k++) {
            int y = yw + k;
            while (y >= ny) y -= ny;
            const uint32_t* row = P + (size_t)y * NW;
            const uint32_t head = row[0];
#pragma unroll
            for (int w = 0; w < WPL; w++) {
                const uint32_t v = __builtin_amdgcn_alignbit(row[ib[w]], row[ia[w]], sh[w]);
                R[k][w] = low[w] == 32u ? v : (v & ((1u << low[w]) - 1u)) | (head << low[w]);
            }
        }
    }
    tw_generations<WPL, K, G, NWAVES, false>(R, Rp, hs, lane, wv, gens);
#pragma unroll
    for (int k = 0; k < K; k++) {
        const int r = wv * K + k - G, y = band * OUT + r;  // output row of the block, of the field
        if (r < 0 || r >= OUT || y >= ny) continue;
        uint32_t* row = Q + (size_t)y * NW;
#pragma unroll
        for (int w = 0; w < WPL; w++) {
            const int lw = WPL * lane + w;
            if (lw >= 1 && lw <= OUTW && g0 + w < NW) row[g0 + w] = R[k][w];
        }
    }
}

// Window variants.  Few rows a wave make a generation short (about 0.07 + 0.08 K us for a block
// alone on its CU, whose waves meet at a barrier each generation), many make the 2G rows that
// a block repeats cheap, and G spreads the 4.5 us that a launch costs.
struct WinVariant {
    const char* name;
    void (*kernel)(const uint32_t*, uint32_t*, int, int, int, int, int);
    int k, g, nwaves;
};
#define WIN(K, G, NWAVES) {"win k" #K " g" #G " w" #NWAVES, k_step_win<1, K, G, NWAVES>, K, G, NWAVES}
static const WinVariant kWin[] = {WIN(4, 24, 16), WIN(6, 24, 16), WIN(6, 16, 16), WIN(8, 24, 16), WIN(8, 16, 16),
                                  WIN(12, 16, 16)};
constexpr int WIN_WORDS = 62;  // words of a row that a window stores
constexpr int TB_K = 10, TB_G = 4, TB_WAVES = 16;  // "tb k10 g4 w16"

typedef void (*tw_io_kernel)(const uint8_t*, const uint32_t*, uint32_t*, uint8_t*, uint8_t*, int, int, int, int);
struct TwVariant {
    const char* name;
    void (*kernel)(const uint32_t*, uint32_t*, int, int, int, int);
    int k, g, nwaves, wpl;  // wpl: words per lane; a wave spans a row of 64 * wpl words
    // the first launch of a call reading the uint8 field, and the last one writing both
    // uint8 buffers (k_step_tw_io)
    tw_io_kernel kin, kout;
};
#define TW_IO(WPL, K, G, NWAVES) k_step_tw_io<WPL, K, G, NWAVES, true, false>, k_step_tw_io<WPL, K, G, NWAVES, false, true>

static const TwVariant kTw[] = {
    // 32 output rows per block: 256 blocks fill 256 CUs at 8192 rows
    {"tw4 k3 g8 w16", k_step_tw<4, 3, 8, 16>, 3, 8, 16, 4, TW_IO(4, 3, 8, 16)},
    {"tw4 k4 g8 w12", k_step_tw<4, 4, 8, 12>, 4, 8, 12, 4, TW_IO(4, 4, 8, 12)},
    {"tw2 k3 g8 w16", k_step_tw<2, 3, 8, 16>, 3, 8, 16, 2, TW_IO(2, 3, 8, 16)},
    {"tw1 k3 g8 w16", k_step_tw<1, 3, 8, 16>, 3, 8, 16, 1, TW_IO(1, 3, 8, 16)},
};

}  // namespace golbits

namespace {

// `gens` generations from P[*cur] in windows of variant v
int run_win(appfis_ctx* ctx, const golbits::WinVariant& v, uint32_t* const P[2], int* cur, int nx, int ny, int gens,
            int* launches)
{
    const int NW = (nx + 31) / 32, tiles_x = (int)ceil_div(NW, golbits::WIN_WORDS);
    const unsigned bands = ceil_div(ny, v.nwaves * v.k - 2 * v.g);
    *launches = 0;
    for (int done = 0; done < gens;) {
        const int n = std::min(gens - done, v.g);
        hipLaunchKernelGGL(v.kernel, dim3(bands * tiles_x), dim3(64 * v.nwaves), 0, ctx->stream, P[*cur], P[*cur ^ 1],
                           nx, NW, ny, tiles_x, n);
        APPFIS_LAUNCH_CHECK();
        *cur ^= 1;
        done += n;
        ++*launches;
    }
    return APPFIS_OK;
}

// The window variant for `gens` generations of an nx x ny board, by the cost that its table
// states: blocks that share a CU take about 0.8 of their times' sum.  Measured (48 generations,
// us; k4 g24, k6 g24, k6 g16, k8 g24, k8 g16, k12 g16): 1000 x 1000 23 30 34 37 43 56; 3000 x 3000
// 34 30 34 37 42 57; 8191 x 8191 139 88 79 86 71 92; 16384 x 16384 457 247 199 201 196 171.
double win_blocks(const golbits::WinVariant& v, int nx, int ny)
{
    return (double)ceil_div((nx + 31) / 32, golbits::WIN_WORDS) * ceil_div(ny, v.nwaves * v.k - 2 * v.g);
}
double win_cost(const appfis_ctx* ctx, const golbits::WinVariant& v, int nx, int ny, int gens)
{
    const double cus = ctx->num_cu > 0 ? ctx->num_cu : 256, blocks = win_blocks(v, nx, ny);
    const double load = blocks <= cus ? 1.0 : 0.8 * std::ceil(blocks / cus);
    return 4.5 * ceil_div(gens, v.g) + gens * (0.07 + 0.0775 * v.k) * load;
}
const golbits::WinVariant& win_for(const appfis_ctx* ctx, int nx, int ny, int gens)
{
    const golbits::WinVariant* best = nullptr;
    double least = 0.0;
    for (const golbits::WinVariant& v : golbits::kWin) {
        const double cost = win_cost(ctx, v, nx, ny, gens);
        if (!best || cost < least) {
            best = &v;
            least = cost;
        }
    }
    return *best;
}

// `gens` generations from P[*cur] one by one
int run_step(appfis_ctx* ctx, uint32_t* const P[2], int* cur, int NW, int ny, int gens, int* launches)
{
    using namespace golbits;
    const unsigned nitems = (unsigned)NW * ceil_div(ny, KROWS);
    for (int g = 0; g < gens; g++) {
        hipLaunchKernelGGL(k_step<KROWS>, dim3(ceil_div(nitems, 256)), dim3(256), 0, ctx->stream, P[*cur], P[*cur ^ 1],
                           NW, ny, nitems);
        APPFIS_LAUNCH_CHECK();
        *cur ^= 1;
    }
    *launches = gens;
    return APPFIS_OK;
}

// Whether `gens` generations of a board of whole words run faster one by one than in windows of v.
// One takes 2.9 us and its words' traffic, up to ten times that where rows of few words leave a
// wave's lanes far apart; a window launch of several blocks to a CU loads and stores 2.2 us longer
// for each.  us a call, one by one / windows: 64 x 10^6 2 generations 90 / 146, 30 601 / 678; 512 x
// 131072 2 46.5 / 56.7, 4 57.8 / 62.2, 6 69.1 / 67.9; 96 x 96 2 10.7 / 11.9, 4 16.6 / 12.9.
bool step_faster(const appfis_ctx* ctx, const golbits::WinVariant& v, int nx, int ny, int gens)
{
    const double cus = ctx->num_cu > 0 ? ctx->num_cu : 256, NW = nx / 32;
    const double step = 2.9 + 1.5e-6 * NW * ny * std::max(1.0, 10.0 / NW);
    const double more = std::ceil(win_blocks(v, nx, ny) / cus) - 1.0;
    return gens * step < win_cost(ctx, v, nx, ny, gens) + ceil_div(gens, v.g) * 2.2 * more;
}

// `gens` generations from P[*cur] with k_step_tb, rows spread over NW / 64 waves
int run_tb(appfis_ctx* ctx, uint32_t* const P[2], int* cur, int NW, int ny, int gens, int* launches)
{
    using namespace golbits;
    const int WX = NW / 64, OUT = TB_WAVES / WX * TB_K - 2 * TB_G;
    *launches = 0;
    for (int done = 0; done < gens;) {
        const int n = std::min(gens - done, TB_G);
        hipLaunchKernelGGL((k_step_tb<TB_K, TB_G, TB_WAVES>), dim3(ceil_div(ny, OUT)), dim3(64 * TB_WAVES), 0,
                           ctx->stream, P[*cur], P[*cur ^ 1], NW, ny, WX, OUT, n);
        APPFIS_LAUNCH_CHECK();
        *cur ^= 1;
        done += n;
        ++*launches;
    }
    return APPFIS_OK;
}

// a row is whole waves, a divisor of the block's, and the rows left hold more than the halo
bool tb_fits(int nx)
{
    using namespace golbits;
    const int WX = nx / 2048;
    return nx % 2048 == 0 && WX <= TB_WAVES && TB_WAVES % WX == 0 && TB_WAVES / WX * TB_K > 2 * TB_G;
}

int tw_out(const golbits::TwVariant& v) { return v.nwaves * v.k - 2 * v.g; }

// `gens` generations from P[*cur] with full-row variant v (G per launch)
int run_tw(appfis_ctx* ctx, const golbits::TwVariant& v, uint32_t* const P[2], int* cur, int NW, int ny, int gens)
{
    const int OUT = tw_out(v);
    for (int done = 0; done < gens;) {
        const int n = std::min(gens - done, v.g);
        hipLaunchKernelGGL(v.kernel, dim3(ceil_div(ny, OUT)), dim3(64 * v.nwaves), 0, ctx->stream, P[*cur], P[*cur ^ 1],
                           NW, ny, OUT, n);
        APPFIS_LAUNCH_CHECK();
        *cur ^= 1;
        done += n;
    }
    return APPFIS_OK;
}

size_t packed_bytes(int nx, int ny) { return ((size_t)((nx + 31) / 32) * ny * 4 + 255) / 256 * 256; }

}  // namespace

bool gol_bits_workspace(appfis_ctx* ctx, int nx, int ny)
{
    if (ensure_work(ctx, 2 * packed_bytes(nx, ny)) == APPFIS_OK) return true;
    (void)hipGetLastError();  // an allocation that failed is no error of the launches that follow
    return false;
}

// Runs `gens` >= 1 generations of the nx x ny periodic field (nx >= 32) held in buf0; see the
// file comment for what the two buffers hold on return.  Two blocked forms advance the packed
// field: windows (k_step_win) for any width, their shape chosen by win_for, and, where a wave
// spans the row (nx = 2048, 4096 or 8192), full-row waves (k_step_tw), which the tuner times
// against the window (at 8192 x 8192 63 us for 48 generations against 69, at 2048 x 2048 31
// against 24).  With full-row waves and two or more generations, all of them run in their
// launches (at least two), the first reading the uint8 field and the last writing both uint8
// buffers; otherwise k_pack packs the field, generations 1 .. gens-1 run blocked, or one by one
// where step_faster says so, and the last one runs fused with the unpacking (k_step_unpack), so
// that generation gens-1 is still at hand.
int gol_bits_run(appfis_ctx* ctx, uint8_t* b0, uint8_t* b1, int nx, int ny, int gens, int force)
{
    const int NW = (nx + 31) / 32;
    const int ntw = (int)(sizeof(golbits::kTw) / sizeof(golbits::kTw[0]));
    const int nwin = (int)(sizeof(golbits::kWin) / sizeof(golbits::kWin[0]));
    const auto fits = [&](int i) { return nx % 32 == 0 && NW == 64 * golbits::kTw[i].wpl; };
    if (force >= 0) {
        APPFIS_REQUIRE(nx >= 32, "gol: the bit-packed form needs nx >= 32 (nx = %d)", nx);
        APPFIS_REQUIRE(force <= ntw + nwin, "gol: candidate %d out of range (%d candidates)", force, ntw + nwin + 1);
        APPFIS_REQUIRE(force >= ntw || fits(force), "gol: candidate %s needs nx that its waves span (nx = %d)",
                       golbits::kTw[force].name, nx);
        APPFIS_REQUIRE(force < ntw + nwin || tb_fits(nx), "gol: candidate tb needs nx that its block spans (nx = %d)", nx);
    }
    const size_t half = packed_bytes(nx, ny);
    int st = ensure_work(ctx, 2 * half);
    if (st) return st;
    uint32_t* const P[2] = {(uint32_t*)ctx->work, (uint32_t*)((char*)ctx->work + half)};
    const golbits::WinVariant* win = force >= ntw && force < ntw + nwin ? &golbits::kWin[force - ntw] : nullptr;
    const golbits::TwVariant* tw = force >= 0 && force < ntw ? &golbits::kTw[force] : nullptr;
    if (force < 0) {
        win = &win_for(ctx, nx, ny, gens > 1 ? gens - 1 : 1);
        std::vector<const golbits::TwVariant*> cand;
        std::vector<const char*> names;
        for (int i = 0; i < ntw; i++)
            if (fits(i)) {
                cand.push_back(&golbits::kTw[i]);
                names.push_back(golbits::kTw[i].name);
            }
        if (!cand.empty() && gens > 1) {
            // on the two packed buffers before they hold the field (timing does not depend on
            // the cell values); the window is the rule's for the 48 timed generations
            const golbits::WinVariant& wt = win_for(ctx, nx, ny, 48);
            names.push_back(wt.name);
            const int key[6] = {4, APPFIS_U8, nx, ny, 0, 0};
            int c = 0;
            st = tune_select(ctx, key, (int)names.size(), names.data(),
                             [&](int i) {
                                 int tmp = 0, n = 0;
                                 return i < (int)cand.size() ? run_tw(ctx, *cand[i], P, &tmp, NW, ny, 48)
                                                             : run_win(ctx, wt, P, &tmp, nx, ny, 48, &n);
                             },
                             4, &c);
            if (st) return st;
            if (c < (int)cand.size()) tw = cand[c];
            // The tuner times the generations alone.  In a short call the two launches that the
            // full-row form does without, its first packing the board and its last unpacking it,
            // count for more than its longer generations, where a lane holds one word (2048 x
            // 2048, us a call, full rows / windows: 2 generations 13.9 / 15.3, 16 18.3 / 20.3,
            // 24 23.3 / 22.7; 4096 x 1000, two words: 20.2 / 15.3, 27.5 / 20.5, 33.8 / 22.9).
            else if (cand[0]->wpl == 1 && gens < 20) tw = cand[0];
        }
    }
    uint8_t* buf[2] = {b0, b1};
    if (tw && gens >= 2) {
        // full-row form over two or more launches: the first packs the uint8 field as it
        // loads its window, the last writes generations gens and gens-1 back as uint8
        // (rings included) -- after the first has finished reading b0, which it may
        // overwrite.  Up to G generations: gens-1 in the first launch, 1 in the last;
        // beyond: G per launch, the rest in the last.
        const golbits::TwVariant& v = *tw;
        const int OUT = tw_out(v);
        const dim3 grid(ceil_div((size_t)ny, (size_t)OUT)), block(64 * v.nwaves);
        const int L = gens <= v.g ? 2 : (gens + v.g - 1) / v.g;
        const int first = gens <= v.g ? gens - 1 : v.g;
        const int last = gens - first - (L - 2) * v.g;
        st = ktime_begin(ctx);
        if (st) return st;
        hipLaunchKernelGGL(v.kin, grid, block, 0, ctx->stream, b0, nullptr, P[0], nullptr, nullptr, nx, ny, OUT,
                           first);
        APPFIS_LAUNCH_CHECK();
        int cur = 0;
        for (int l = 1; l < L - 1; l++) {
            hipLaunchKernelGGL(v.kernel, grid, block, 0, ctx->stream, P[cur], P[cur ^ 1], NW, ny, OUT, v.g);
            APPFIS_LAUNCH_CHECK();
            cur ^= 1;
        }
        hipLaunchKernelGGL(v.kout, grid, block, 0, ctx->stream, nullptr, P[cur], nullptr, buf[gens & 1],
                           buf[(gens & 1) ^ 1], nx, ny, OUT, last);
        APPFIS_LAUNCH_CHECK();
        return ktime_end(ctx, L, gens);
    }
    const unsigned pblocks = ceil_div((size_t)NW * ny, 256);
    hipLaunchKernelGGL(golbits::k_pack, dim3(pblocks), dim3(256), 0, ctx->stream, b0, P[0], nx, ny, NW);
    APPFIS_LAUNCH_CHECK();
    int cur = 0, launches = 0;
    st = ktime_begin(ctx);
    if (st) return st;
    if (gens > 1) {
        if (!win)
            st = run_tb(ctx, P, &cur, NW, ny, gens - 1, &launches);
        else if (force < 0 && nx % 32 == 0 && step_faster(ctx, *win, nx, ny, gens - 1))
            st = run_step(ctx, P, &cur, NW, ny, gens - 1, &launches);
        else
            st = run_win(ctx, *win, P, &cur, nx, ny, gens - 1, &launches);
        if (st) return st;
    }
    st = ktime_end(ctx, launches, gens - 1);
    if (st) return st;
    // generation gens-1 is in P[cur]: the last generation runs fused with the unpacking
    // of generations gens (into buf[gens % 2]) and gens-1 (the other buffer), rings
    // exchanged
    const int nbands = (ny + golbits::KROWS - 1) / golbits::KROWS;
    const unsigned nitems = (unsigned)NW * (unsigned)nbands;
    hipLaunchKernelGGL(golbits::k_step_unpack<golbits::KROWS>, dim3(ceil_div(nitems, 256)), dim3(256), 0,
                       ctx->stream, P[cur], buf[gens & 1], buf[(gens & 1) ^ 1], nx, NW, ny, nitems);
    APPFIS_LAUNCH_CHECK();
    return APPFIS_OK;
}

extern "C" int appfis_gol_candidates(char* names, int len)
{
    std::string all;
    int n = 0;
    for (const golbits::TwVariant& v : golbits::kTw) all += std::string(v.name) + "\n", n++;
    for (const golbits::WinVariant& v : golbits::kWin) all += std::string(v.name) + "\n", n++;
    all += "tb k10 g4 w16\n";
    if (names && len > 0) snprintf(names, (size_t)len, "%s", all.c_str());
    return n + 1;
}
