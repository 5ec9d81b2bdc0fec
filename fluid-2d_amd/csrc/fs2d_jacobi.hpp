// fs2d_jacobi.hpp -- device pieces shared by the one-grid sweep kernels
// (fs2d_sweeps.hip, fs2d_jacobi.hip) and the batched kernels (fs2d_batch.hip):
// the diffuse division, the relaxation of one cell, and the Jacobi block tile.
#pragma once

#include "fs2d_cells.hpp"
#include "fs2d_internal.hpp"

namespace fs2d {
namespace jac {

__device__ __forceinline__ float sgn(bool neg, float x) { return neg ? -x : x; }

// The divisor of a diffuse solve: d = 1 + 4a, y = RN(1/d), y_lo = RN(1/d - y)
// (so y + y_lo is 1/d to about 2^-48), and lo, the smallest nonzero
// |dividend| the corrected quotient takes (the host's division_floor:
// max(2^-100, d 2^-124), or +inf when d > 2^100).  y2, y2_lo and lo2 are the same
// of the checked quotient (known_quotient): lo2 is 0 for a power of two, whose pair
// is exact for every dividend, but Markstein's step turns -0 into +0, so a field
// with such a divisor that shares a launch with an unchecked one needs its own lo.
struct Divisor {
    float d, y, lo, y_lo, y2, y2_lo, lo2;
};

__host__ __device__ __forceinline__ Divisor divisor_of(const SweepArgs& A) {
    return Divisor{A.denom, A.inv_denom, A.div_lo, A.inv_denom_lo, A.inv_hi2, A.inv_lo2, A.div_lo2};
}

// Dividends outside [lo, 2^100] (zero, tiny, huge, inf, NaN) take the IEEE
// division.  The test is wave-uniform: the common step, where no lane needs
// it, passes one untaken branch.
__device__ __forceinline__ float div_outside(float q, float x, Divisor v) {
    const float ax = fabsf(x);
    const bool out = !(ax >= v.lo && ax <= 0x1p100f);
    if (__builtin_expect(__builtin_amdgcn_ballot_w64(out) != 0, 0)) q = out ? x / v.d : q;
    return q;
}

// x / d correctly rounded.  q1 = RN(x y + RN(x y_lo)) is within 2^-47
// relative of x/d before its rounding, so faithful; Markstein's step from a
// faithful quotient, its remainder exact by FMA, rounds correctly (P.
// Markstein, IBM J. R&D 34(1), 1990; Muller et al., Handbook of
// Floating-Point Arithmetic, FMA-based division), for lo <= |x| <= 2^100.
// Pinned against exact rational arithmetic in tests/test_division.py.
__device__ __forceinline__ float div_rn(float x, Divisor v) {
    const float q1 = __builtin_fmaf(x, v.y, x * v.y_lo);
    return div_outside(__builtin_fmaf(__builtin_fmaf(-q1, v.d, x), v.y, q1), x, v);
}

// x / d for a divisor whose two-product quotient RN(x y2 + RN(x y2_lo)) the
// host has checked to be correctly rounded for every finite dividend from lo2
// up (Brisebarre, Muller and Raina, "Accelerating correctly rounded
// floating-point division when the divisor is known in advance", IEEE Trans.
// Computers 53(8), 2004; the check is two_product_quotient).  With y2_lo > 0
// an infinite dividend gives the infinity IEEE division gives, so one test,
// |x| >= lo2 (false for tiny, subnormal and NaN), guards it.
__device__ __forceinline__ float div_rn_checked(float x, Divisor v) {
    float q = __builtin_fmaf(x, v.y2, x * v.y2_lo);
    const bool out = !(fabsf(x) >= v.lo2);
    if (__builtin_expect(__builtin_amdgcn_ballot_w64(out) != 0, 0)) q = out ? x / v.d : q;
    return q;
}

// The update of one cell; operand order as in src/fluid_solver_cpu.cpp:107-108
// (diffuse: N + S + W + E) and :199-200 (pressure: d + E + W + S + N).
__device__ __forceinline__ float relax(int kind, float b, float n, float s, float w, float e, float a, Divisor dv) {
    if (kind == SWEEP_DIFFUSE) return div_rn(b + a * (((n + s) + w) + e), dv);
    return ((((b + e) + w) + s) + n) / 4.0f;
}

// ===================== Gauss-Seidel tile hyperplane ======================
// CHECKED: the diffuse quotient is div_rn_checked (a divisor the host checked).
template <int KIND, bool CHECKED = false>
__device__ __forceinline__ float relax_k(float b, float n, float s, float w, float e, float a, Divisor dv) {
    if (KIND == SWEEP_DIFFUSE) {
        const float x = b + a * (((n + s) + w) + e);
        return CHECKED ? div_rn_checked(x, dv) : div_rn(x, dv);
    }
    return ((((b + e) + w) + s) + n) / 4.0f;
}

// The same update with the diffuse quotient taken on the fast path only: the
// wave's lanes whose dividend the fast path does not cover are ORed into bad
// (a ballot, no branch), and the caller redoes its steps with relax_k when bad
// is nonzero.  Pressure updates have no division and leave bad alone.
template <int KIND, bool CHECKED>
__device__ __forceinline__ float relax_fast(float b, float n, float s, float w, float e, float a, Divisor dv,
                                            unsigned long long& bad) {
    if (KIND == SWEEP_DIFFUSE) {
        const float x = b + a * (((n + s) + w) + e);
        if (CHECKED) {
            bad |= __builtin_amdgcn_ballot_w64(!(fabsf(x) >= dv.lo2));
            return __builtin_fmaf(x, dv.y2, x * dv.y2_lo);
        }
        const float ax = fabsf(x);
        bad |= __builtin_amdgcn_ballot_w64(!(ax >= dv.lo && ax <= 0x1p100f));
        const float q1 = __builtin_fmaf(x, dv.y, x * dv.y_lo);
        return __builtin_fmaf(__builtin_fmaf(-q1, dv.d, x), dv.y, q1);
    }
    return ((((b + e) + w) + s) + n) / 4.0f;
}

__device__ __forceinline__ float lane_west(float x) {  // lane l receives lane l - 1
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x138, 0xf, 0xf, false));
}
__device__ __forceinline__ float lane_east(float x) {  // lane l receives lane l + 1
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x130, 0xf, 0xf, false));
}

// ===================== Jacobi, block tiles ===============================
// A block of NW waves relaxes a region of NW RPW rows x 64 columns m times (m <=
// kTileMaxSweeps, a run-time count): wave w holds rows RPW w .. of the iterate
// and of the right-hand side in registers, lane l column l.  West and east come
// from lanes l -+ 1 by a full-wave DPP shift folded into the additions, north
// and south from the wave's own rows or, at its first and last row, through
// LDS: each sweep starts with every wave storing those two rows and one barrier
// (two buffers, used in turn).
//
// Against one wave per tile (48 rows in one wave's registers) no halo lies between
// waves, and a tile has 8 times the waves, each an eighth of the chain: a launch of
// 8 sweeps of 258 x 258 cells took 18.6 us and takes 5.5.  The measured shapes
// and what bounds them are in fs2d_jacobi.hip.
//
// Rows live in RPW + 1 register slots: a sweep down the rows writes row r where
// row r - 1 was, the next sweep, up the rows, writes it back, so no sweep copies
// registers.  Tiles never start outside the grid: the ring is a region's own
// first or last row or column there, and needs no halo.  A ring neighbour is the
// stored ring in a launch's first sweep, and the ring of the sweep before, the
// sign-adjusted value of the cell itself, after that.
constexpr int kTileMaxSweeps = 8, kTileCols = 64;

// What a tile loads.  TILE_STORED: the iterate and the right-hand side b.  The first
// launch of a solve can form b from what b's own pass would read, and store it for the
// launches after it, so that pass's launch and its reads and writes fall away:
//   TILE_SOURCES     b and the iterate are src + scale s0 (src_x + dt s, a step's source
//                    term); ring cells of the iterate are src's
//   TILE_DIVERGENCE  b is the divergence scale (((s0E - s0W) + s1S) - s1N) of a velocity
//                    s0, s1; the iterate starts as zero
// A cell of the halo is formed by every tile that holds it, the same each time.
//   TILE_GRADIENT    stored, and after the sweeps (a pressure solve's last) the tile
//                    subtracts the pressure's gradient from gu and gv in place, as
//                    cells::gradient, which saves the pass that would read the pressure
//                    back.  Tiles are placed for m + 1 sweeps then.  Never in a launch
//                    that also reads the velocity's halo (TILE_DIVERGENCE).
enum TileLoad : int { TILE_STORED = 0, TILE_SOURCES = 1, TILE_DIVERGENCE = 2, TILE_GRADIENT = 3 };

struct TileJob {
    const float *src, *b;
    float* dst;
    const float *s0, *s1;  // TILE_SOURCES, TILE_DIVERGENCE
    float scale;
    float* b_out;
    float *gu, *gv;        // TILE_GRADIENT
    float h;
    unsigned* speed_slot;  // takes the largest speed of the result if not null (cells::fold_speed)
    int R, P, m;
    bool zero;  // the iterate starts as zero (src is not read)
    float a;
    Divisor dv;
    Ring rg;
    int gi0, gj0;            // grid cell of the region's first cell
    int ilo, ihi, jlo, jhi;  // cells written
};

// Tiles of regions `extent` cells long that cover R cells, m of each end of a
// region lost to the sweeps except where the grid ends.
__host__ __device__ inline int tile_count(int R, int extent, int m) {
    return R <= extent ? 1 : (R - 2 * m + extent - 2 * m - 1) / (extent - 2 * m);
}
// The region and output range of tile (ty, tx) of tiles_y x tiles_x (tile_count)
// with H x kTileCols regions; the last tile is moved back to end with the grid.
__device__ __forceinline__ void tile_place(TileJob& t, int H, int ty, int tx, int tiles_y, int tiles_x) {
    const int sy = H - 2 * t.m, sx = kTileCols - 2 * t.m;
    t.gi0 = t.R <= H ? 0 : min(ty * sy, t.R - H);
    t.gj0 = t.R <= kTileCols ? 0 : min(tx * sx, t.R - kTileCols);
    t.ilo = ty == 0 ? 1 : ty * sy + t.m;
    t.ihi = ty == tiles_y - 1 ? t.R - 2 : ty * sy + H - 1 - t.m;
    t.jlo = tx == 0 ? 1 : tx * sx + t.m;
    t.jhi = tx == tiles_x - 1 ? t.R - 2 : tx * sx + kTileCols - 1 - t.m;
}

enum TileKind : int { TILE_DIFFUSE = 0, TILE_PRESSURE = 1, TILE_DIFFUSE_CHECKED = 2 };

// The update of one cell.  A checked divisor's quotient is taken at once; where
// some lane's dividend lies below its range, the IEEE division replaces it.
// Zeros lie below it too, but their quotient is exact.
template <int KIND>
__device__ __forceinline__ float relax_tile(float b, float n, float s, float w, float e, float a, const Divisor& dv) {
    if constexpr (KIND == TILE_PRESSURE) return ((((b + e) + w) + s) + n) / 4.0f;
    const float x = b + a * (((n + s) + w) + e);
    if constexpr (KIND == TILE_DIFFUSE) return div_rn(x, dv);
    float q = __builtin_fmaf(x, dv.y2, x * dv.y2_lo);
    const bool low = !(fabsf(x) >= dv.lo2);
    if (__builtin_expect(__builtin_amdgcn_ballot_w64(low) != 0, 0)) {
        const bool bad = low && x != 0.f;
        if (__builtin_amdgcn_ballot_w64(bad) != 0) q = bad ? x / dv.d : q;
    }
    return q;
}

// Where a region holds the ring.  A region of a grid no smaller than it has the ring
// as its own first or last row (ROWS 1) and its first (COLS 1) or last column (COLS 2),
// so the cells beside the ring are known rows and lanes: two rows of a tile's eighth
// and one neighbour a row are selected, and the other neighbour stays folded into its
// addition.  2 / 3: anywhere (a grid smaller than the region, or one with both columns
// in it), tested by index in every row.
// ex: 4 NW kTileCols floats of LDS.
template <int RPW, int NW, int KIND, int LOAD, int ROWS, int COLS>
__device__ __forceinline__ void jacobi_tile(const TileJob& t, float* __restrict__ ex) {
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int R = t.R, P = t.P, n = R - 2, i0 = t.gi0 + wave * RPW, gj = t.gj0 + lane;
    const int cj = min(gj, R - 1);  // a grid narrower than the region
    float X[RPW + 1], B[RPW];
    if constexpr (LOAD == TILE_STORED || LOAD == TILE_GRADIENT) {
#pragma unroll
        for (int r = 0; r < RPW; ++r) X[r + 1] = t.zero ? 0.f : t.src[(size_t)min(i0 + r, R - 1) * P + cj];
#pragma unroll
        for (int r = 0; r < RPW; ++r) B[r] = t.b[(size_t)min(i0 + r, R - 1) * P + cj];
    } else {
        if constexpr (LOAD == TILE_SOURCES) {
#pragma unroll
            for (int r = 0; r < RPW; ++r) X[r + 1] = t.src[(size_t)min(i0 + r, R - 1) * P + cj];
#pragma unroll
            for (int r = 0; r < RPW; ++r) B[r] = t.s0[(size_t)min(i0 + r, R - 1) * P + cj];
#pragma unroll
            for (int r = 0; r < RPW; ++r) {
                B[r] = X[r + 1] + t.scale * B[r];
                const bool ring = (ROWS && (i0 + r < 1 || i0 + r > n)) || (COLS && (gj < 1 || gj > n));
                X[r + 1] = ring ? X[r + 1] : B[r];
            }
        } else {
            // the region's first and last rows and lanes lack a neighbour; they are
            // ring or lost to the first sweep
            float V[RPW + 2];
#pragma unroll
            for (int r = 0; r < RPW + 2; ++r) V[r] = t.s1[(size_t)max(min(i0 + r - 1, R - 1), 0) * P + cj];
#pragma unroll
            for (int r = 0; r < RPW; ++r) B[r] = t.s0[(size_t)min(i0 + r, R - 1) * P + cj];
#pragma unroll
            for (int r = 0; r < RPW; ++r) {
                B[r] = t.scale * (((lane_east(B[r]) - lane_west(B[r])) + V[r + 2]) - V[r]);
                X[r + 1] = 0.f;
            }
        }
        if (gj >= t.jlo && gj <= t.jhi) {
#pragma unroll
            for (int r = 0; r < RPW; ++r)
                if (i0 + r >= t.ilo && i0 + r <= t.ihi) t.b_out[(size_t)(i0 + r) * P + gj] = B[r];
        }
    }

    const float a = t.a;
    const Divisor dv = t.dv;
    const Ring rg = t.rg;
    const bool top = t.gi0 == 0 && wave == 0, bottom = t.gi0 + NW * RPW == R && wave == NW - 1;  // ROWS 1
    // row r of sweep s, from its own value c and its neighbours above and below
    auto row = [&](int s, int r, float c, float north, float south) {
        float west = lane_west(c), east = lane_east(c);
        if (ROWS == 1 && s > 0) {
            if (r == 1) north = top ? sgn(rg.neg_tb, c) : north;
            if (r == RPW - 2) south = bottom ? sgn(rg.neg_tb, c) : south;
        }
        if (COLS == 1 && s > 0) west = lane == 1 ? sgn(rg.neg_lr, c) : west;
        if (COLS == 2 && s > 0) east = lane == kTileCols - 2 ? sgn(rg.neg_lr, c) : east;
        if (ROWS == 2 && s > 0) {
            const int gi = i0 + r;  // the same in all lanes
            const float m = sgn(rg.neg_tb, c);
            north = gi == 1 ? m : north;
            south = gi == n ? m : south;
        }
        if (COLS == 3 && s > 0) {
            const float m = sgn(rg.neg_lr, c);
            west = gj == 1 ? m : west;
            east = gj == n ? m : east;
        }
        return relax_tile<KIND>(B[r], north, south, west, east, a, dv);
    };
    auto exchange = [&](int s, float first, float last, float& above, float& below) {
        float* const e = ex + (s & 1) * NW * 2 * kTileCols + lane;
        e[(2 * wave) * kTileCols] = first;
        e[(2 * wave + 1) * kTileCols] = last;
        __syncthreads();
        above = e[(2 * max(wave - 1, 0) + 1) * kTileCols];
        below = e[(2 * min(wave + 1, NW - 1)) * kTileCols];
    };
    // rows in slots 1 .. RPW -> slots 0 .. RPW - 1, and back
    auto down = [&](int s) {
        float above, below;
        exchange(s, X[1], X[RPW], above, below);
#pragma unroll
        for (int r = 0; r < RPW; ++r)
            X[r] = row(s, r, X[r + 1], r > 0 ? X[r] : above, r + 1 < RPW ? X[r + 2 <= RPW ? r + 2 : RPW] : below);
    };
    auto up = [&](int s) {
        float above, below;
        exchange(s, X[0], X[RPW - 1], above, below);
#pragma unroll
        for (int r = RPW - 1; r >= 0; --r)
            X[r + 1] = row(s, r, X[r], r > 0 ? X[r > 0 ? r - 1 : 0] : above, r + 1 < RPW ? X[r + 1] : below);
    };
    int s = 0;
    for (; s + 1 < t.m; s += 2) {
        down(s);
        up(s + 1);
    }
    if (s < t.m) {
        down(s);
#pragma unroll
        for (int r = RPW - 1; r >= 0; --r) X[r + 1] = X[r];
    }

    if constexpr (LOAD == TILE_GRADIENT) {
        float above, below, speed = 0.f;
        exchange(t.m, X[1], X[RPW], above, below);
        const bool own = gj >= t.jlo && gj <= t.jhi;
#pragma unroll
        for (int r = 0; r < RPW; ++r) {
            const int gi = i0 + r;
            if (gi < t.ilo || gi > t.ihi) continue;  // the same in all lanes
            const float c = X[r + 1];
            float pn = r > 0 ? X[r] : above, ps = r + 1 < RPW ? X[r + 2 <= RPW ? r + 2 : RPW] : below;
            float pw = lane_west(c), pe = lane_east(c);
            if (ROWS) {  // the pressure's ring continues it
                pn = gi == 1 ? c : pn;
                ps = gi == n ? c : ps;
            }
            if (COLS) {
                pw = gj == 1 ? c : pw;
                pe = gj == n ? c : pe;
            }
            if (own) {
                const size_t g = (size_t)gi * P + gj;
                const float un = t.gu[g] - 0.5f * (pe - pw) / t.h;
                const float vn = t.gv[g] - 0.5f * (ps - pn) / t.h;
                t.gu[g] = un;
                t.gv[g] = vn;
                if (ROWS || COLS) {
                    cells::write_ring(t.gu, gi, gj, un, R, P, Ring{false, true});
                    cells::write_ring(t.gv, gi, gj, vn, R, P, Ring{true, false});
                }
                speed = cells::fold_speed(speed, un, vn);
            }
        }
        if (t.speed_slot) {
            for (int off = 32; off > 0; off >>= 1) speed = fmaxf(speed, __shfl_xor(speed, off));
            if (lane == 0) atomicMax(t.speed_slot, __float_as_uint(speed));
        }
    }

    if (gj < t.jlo || gj > t.jhi) return;
    float* __restrict__ dst = t.dst;
#pragma unroll
    for (int r = 0; r < RPW; ++r) {
        const int gi = i0 + r;
        if (gi < t.ilo || gi > t.ihi) continue;  // the same in all lanes
        const float v = X[r + 1];
        const size_t g = (size_t)gi * P + gj;
        dst[g] = v;
        if (!ROWS && !COLS) continue;
        // the ring beside the cell
        const float tb = sgn(rg.neg_tb, v), lr = sgn(rg.neg_lr, v);
        const float cn = 0.5f * (tb + lr);
        if (gi == 1) dst[g - P] = tb;
        if (gi == n) dst[g + P] = tb;
        if (gj == 1) dst[g - 1] = lr;
        if (gj == n) dst[g + 1] = lr;
        if (gi == 1 && gj == 1) dst[g - P - 1] = cn;
        if (gi == 1 && gj == n) dst[g - P + 1] = cn;
        if (gi == n && gj == 1) dst[g + P - 1] = cn;
        if (gi == n && gj == n) dst[g + P + 1] = cn;
    }
}

template <int RPW, int NW, int KIND, int LOAD>
__device__ __forceinline__ void jacobi_tile_any(const TileJob& t, float* __restrict__ ex) {
    const bool left = t.gj0 == 0, right = t.gj0 + kTileCols >= t.R;
    if (t.R < NW * RPW || (left && right)) {
        jacobi_tile<RPW, NW, KIND, LOAD, 2, 3>(t, ex);
    } else if (t.gi0 == 0 || t.gi0 + NW * RPW == t.R) {
        if (left) jacobi_tile<RPW, NW, KIND, LOAD, 1, 1>(t, ex);
        else if (right) jacobi_tile<RPW, NW, KIND, LOAD, 1, 2>(t, ex);
        else jacobi_tile<RPW, NW, KIND, LOAD, 1, 0>(t, ex);
    } else {
        if (left) jacobi_tile<RPW, NW, KIND, LOAD, 0, 1>(t, ex);
        else if (right) jacobi_tile<RPW, NW, KIND, LOAD, 0, 2>(t, ex);
        else jacobi_tile<RPW, NW, KIND, LOAD, 0, 0>(t, ex);
    }
}

// Blocks are dealt round-robin to the 8 XCDs; the first 8 * floor(nb / 8)
// are renumbered so that each XCD walks a contiguous run of tiles (rows of
// tiles in order), whose shared halo rows and columns then meet in its L2.
__device__ __forceinline__ int xcd_block(int b, int nb) {
    const int full = nb - nb % 8;
    return b < full ? (b % 8) * (full / 8) + b / 8 : b;
}

}  // namespace jac
}  // namespace fs2d
