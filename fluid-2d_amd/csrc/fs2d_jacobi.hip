// fs2d_jacobi.hip -- Jacobi sweeps of one to three fields of a grid, block tiles
// (fs2d_jacobi.hpp).
#include "fs2d_jacobi.hpp"

namespace fs2d {
namespace {

using namespace jac;

struct TileSet {
    SweepArgs a[3];
    const float* src[3];
    float* dst[3];
    JacobiFirst first;
    JacobiLast last;
    int m, zero, tiles_x, tiles_y;
};

// Block: tile blockIdx.x of field blockIdx.y.
template <int RPW, int NW, int KIND, int LOAD>
__global__ __launch_bounds__(64 * NW) void k_jacobi_tile(TileSet S) {
    __shared__ float ex[4 * NW * kTileCols];
    const int f = blockIdx.y, b = xcd_block(blockIdx.x, gridDim.x);
    const SweepArgs& A = S.a[f];
    TileJob t;
    t.src = S.src[f];
    t.dst = S.dst[f];
    t.b = A.b;
    t.R = A.R;
    t.P = A.P;
    t.m = S.m;
    t.zero = S.zero != 0;
    t.a = A.a;
    t.dv = divisor_of(A);
    t.rg = A.ring;
    t.s0 = S.first.s0[f];
    t.s1 = S.first.s1;
    t.scale = S.first.scale;
    t.b_out = S.first.b[f];
    t.gu = S.last.u;
    t.gv = S.last.v;
    t.h = S.last.h;
    t.speed_slot = S.last.slots ? S.last.slots + (blockIdx.x % kSpeedSlots) * kSlotStride : nullptr;
    t.m += LOAD == TILE_GRADIENT;
    tile_place(t, NW * RPW, b / S.tiles_x, b % S.tiles_x, S.tiles_y, S.tiles_x);
    t.m = S.m;
    jacobi_tile_any<RPW, NW, KIND, LOAD>(t, ex);
}

template <int RPW, int NW, int KIND, int FIRST>
void launch_kind(hipStream_t s, const TileSet& S, dim3 grid, dim3 block) {
    if (S.first.any) hipLaunchKernelGGL((k_jacobi_tile<RPW, NW, KIND, FIRST>), grid, block, 0, s, S);
    else hipLaunchKernelGGL((k_jacobi_tile<RPW, NW, KIND, TILE_STORED>), grid, block, 0, s, S);
}

template <int RPW, int NW>
hipError_t launch(hipStream_t s, TileSet& S, int fields, int kind) {
    const int R = S.a[0].R;
    const int margin = S.m + (S.last.u != nullptr);
    S.tiles_y = tile_count(R, NW * RPW, margin);
    S.tiles_x = tile_count(R, kTileCols, margin);
    const dim3 grid(S.tiles_x * S.tiles_y, fields), block(64 * NW);
    if (S.last.u) hipLaunchKernelGGL((k_jacobi_tile<RPW, NW, TILE_PRESSURE, TILE_GRADIENT>), grid, block, 0, s, S);
    else if (kind == TILE_PRESSURE) launch_kind<RPW, NW, TILE_PRESSURE, TILE_DIVERGENCE>(s, S, grid, block);
    else if (kind == TILE_DIFFUSE_CHECKED) launch_kind<RPW, NW, TILE_DIFFUSE_CHECKED, TILE_SOURCES>(s, S, grid, block);
    else launch_kind<RPW, NW, TILE_DIFFUSE, TILE_SOURCES>(s, S, grid, block);
    return hipGetLastError();
}

}  // namespace

// Rows of a tile's region (it is 64 columns wide).  Measured, one launch of 8
// sweeps (us; 3 fields of a diffuse / 1 field of pressure; before: one wave per tile):
//   rows      R = 130      258        514         1026        2050         4098
//   32 (4x8)  5.9 / 5.5  6.6 / 5.5  10.8 / 6.7  22.8 / 9.7  70.4 / 22.8  290 / 72.5
//   48 (6x8)  7.4 / 7.0  7.3 / 6.9  11.0 / 6.9  19.0 / 9.1  52.2 / 18.9  206 / 51.6
//   64 (8x8)  9.0 / 8.2  9.1 / 8.3  11.9 / 8.2  19.6 / 10.1 49.5 / 18.6  189 / 45.8
//   96 (12x8) 12.2 / 11.2 12.2 / 11.4 12.8 / 11.6 21.6 / 12.6 47.2 / 22.4 176 / 46.2
//   before    85.5 / 18.4 86.1 / 18.6 87.2 / 18.8 87.5 / 19.1 150 / 28.9  373 / 62.7
// Few cells: the launch is a chain of sweeps, and fewer rows a wave are a shorter
// one.  Many: each 64-column region spends 16 columns and 16 rows on its halo at 8
// sweeps, so taller is better until too few blocks are left.  At 4098 x 4098, by
// counters, the three fields' launch executes 9.2 VALU operations a cell-sweep of its
// regions, 14.7 a written one, at 82 % of the issue slots, and moves 0.66 GB, 3.6 TB/s:
// issue bounds it, and the halo in it.  A pressure launch executes 9.6 a written
// cell-sweep and moves 0.21 GB in 41 to 51 us, about a copy's rate.
// (These were taken before tiles at the grid's edge knew their ring rows and lanes,
// which took 3 % off a step at 4098 and at 203 and moves no line.)
// Two or four columns a lane (less halo) measured slower at every size: 184 and
// 183 us here, 25 and 31 against 19 us at 1026.
static int tile_rows(long cells) { return cells < 500000 ? 32 : (cells < 8000000 ? 48 : 96); }

hipError_t launch_jacobi_tiles(hipStream_t s, const SweepSet& set, const float* const* src, float* const* dst,
                               int zero_src, int m, const JacobiFirst* first, const JacobiLast* last) {
    if (last && (first || zero_src || set.count != 1 || set.a[0].kind != SWEEP_PRESSURE)) return hipErrorInvalidValue;
    if (m < 1 || m > kTileMaxSweeps || set.count < 1 || set.count > 3) return hipErrorInvalidValue;
    TileSet S{};
    bool checked = true;
    for (int f = 0; f < set.count; ++f) {
        S.a[f] = set.a[f];
        checked = checked && S.a[f].div_checked;
        S.src[f] = src[f];
        S.dst[f] = dst[f];
    }
    if (first) S.first = *first;
    if (last) S.last = *last;
    S.m = m;
    S.zero = zero_src;
    const int kind = set.a[0].kind == SWEEP_PRESSURE ? TILE_PRESSURE : (checked ? TILE_DIFFUSE_CHECKED : TILE_DIFFUSE);
    switch (tile_rows(static_cast<long>(set.count) * set.a[0].R * set.a[0].R)) {
        case 32: return launch<4, 8>(s, S, set.count, kind);
        case 48: return launch<6, 8>(s, S, set.count, kind);
        default: return launch<12, 8>(s, S, set.count, kind);
    }
}

}  // namespace fs2d
