// fs2d_mg.hip -- geometric multigrid for a pressure seed (outside
// parity mode): the pressure equation 4 p - sum(nbrs) = b of
// src/fluid_solver_cpu.cpp:196-204 with the continuous ring, on a hierarchy
// of grids whose sides halve.
//
// On a grid coarsened by two the same 5-point stencil holds with the
// right-hand side scaled by 4 (the operator carries h^2), so the coarse
// right-hand side of a cell is the sum of its four fine residuals.  The
// smoother is weighted Jacobi (omega = 4/5 damps the upper half of the 5-point
// spectrum); the correction is interpolated bilinearly (weights 9/16, 3/16,
// 3/16, 1/16 of the four nearest coarse centres).  A ring cell of the continuous
// ring is the value of the interior cell beside it (corners: of the diagonal
// cell), so no kernel here reads one: a neighbour outside is the cell itself.
//
// What bounds it: a V-cycle of a 1024 x 1024 field moves about 80 MB (16 us)
// and was 120 launches of 2 us with gaps as long, 64 of them sweeps of a 4 x 4
// grid.  So
//   * on sides above kMgTailSide each level takes two launches: k_mg_down (two
//     smoothing sweeps, the residual, its restriction) and k_mg_up
//     (correction, two sweeps), a wave per tile with its rows in registers;
//   * the levels below run in one launch of one block (k_mg_tail), with
//     every iterate in LDS and the coarsest grid's sweeps in registers.
// A projection at 1024 x 1024 to 1 % (three V-cycles, their residuals, divergence,
// gradient and the pressure read back to the host): 1.70 -> 0.62 ms; at 64 x 64
// 0.16 ms.  A cycle's launches: down 5.8 and up 6.9 us on average over the sides
// 1024, 512 and 256, the tail from 128 down 43 us, the residual 10 us.
// kMgTailSide is what one block's LDS and registers hold; 4096 sweeps of a
// 125 x 125 coarsest grid take 4.3 ms there, against 14 ms as launches.
#include "fs2d_internal.hpp"
#include "fs2d_jacobi.hpp"

namespace fs2d {
namespace {

using jac::lane_east;
using jac::lane_west;

constexpr int kMgThreads = 256;

__device__ __forceinline__ void write_with_ring(float* g, int i, int j, int n, int P, float v) {
    const size_t o = (size_t)i * P + j;
    g[o] = v;
    if (i == 1) g[o - P] = v;
    if (i == n) g[o + P] = v;
    if (j == 1) g[o - 1] = v;
    if (j == n) g[o + 1] = v;
    if (i == 1 && j == 1) g[o - P - 1] = v;
    if (i == 1 && j == n) g[o - P + 1] = v;
    if (i == n && j == 1) g[o + P - 1] = v;
    if (i == n && j == n) g[o + P + 1] = v;
}

// One cell of a weighted Jacobi sweep.
__device__ __forceinline__ float smoothed(float c, float b, float n, float s, float w, float e, float omega) {
    const float jac = 0.25f * (b + n + s + w + e);
    return c + omega * (jac - c);
}

// One sweep of a level on its own: the coarsest grid where it is too large for
// k_mg_tail (an odd side above kMgTailSide).
__global__ __launch_bounds__(kMgThreads) void k_mg_smooth(const float* __restrict__ src, float* __restrict__ dst,
                                                          const float* __restrict__ b, int R, int P, float omega) {
    const int n = R - 2, i = blockIdx.y + 1, j = blockIdx.x * kMgThreads + threadIdx.x + 1;
    if (j > n) return;
    const size_t o = (size_t)i * P + j;
    const float c = src[o];
    const float nn = i == 1 ? c : src[o - P], ss = i == n ? c : src[o + P];
    const float ww = j == 1 ? c : src[o - 1], ee = j == n ? c : src[o + 1];
    write_with_ring(dst, i, j, n, P, smoothed(c, b[o], nn, ss, ww, ee, omega));
}

// ---- the levels above the tail: a wave per tile of MG_TY rows x 56 columns.
// Lane l holds column 56 tx - 3 + l of the tile's region (4 lanes of halo a
// side keep tiles and coarse cells aligned), rows in registers; each sweep
// leaves one more row and lane a side stale.
constexpr int MG_TY = 16, MG_TX = 56, MG_WAVES = 4;

struct MgStrip {
    int gi0, gj;        // first region row, this lane's column (interior cells are 1 .. n)
    bool left, right;
};

// One smoothing sweep of region rows FROM .. H - 1 - FROM.
template <int H, int FROM, bool EDGE>
__device__ __forceinline__ void mg_sweep(float (&X)[H], const float (&B)[H], const MgStrip& t, int n, float omega) {
    float north = X[FROM - 1];
#pragma unroll
    for (int q = FROM; q < H - FROM; ++q) {
        const float c = X[q];
        float nn = north, ss = X[q + 1], ww = lane_west(c), ee = lane_east(c);
        if (EDGE) {
            const int gi = t.gi0 + q;
            nn = gi == 1 ? c : nn;
            ss = gi == n ? c : ss;
            ww = t.left ? c : ww;
            ee = t.right ? c : ee;
        }
        north = c;
        X[q] = smoothed(c, B[q], nn, ss, ww, ee, omega);
    }
}

template <int H, bool EDGE>
__device__ __forceinline__ void mg_load(float (&X)[H], const float* __restrict__ src, const MgStrip& t, int n, int P) {
    if (EDGE) {
        const int cj = min(max(t.gj, 1), n);
#pragma unroll
        for (int q = 0; q < H; ++q) X[q] = src[(size_t)min(max(t.gi0 + q, 1), n) * P + cj];
    } else {
        const size_t o = (size_t)t.gi0 * P + t.gj;
#pragma unroll
        for (int q = 0; q < H; ++q) X[q] = src[o + (size_t)q * P];
    }
}

// Two sweeps from p (all zero where p is null) into out, and the coarse
// right-hand side bc.
template <bool EDGE>
__device__ __forceinline__ void mg_down(const float* __restrict__ p, float* __restrict__ out,
                                        const float* __restrict__ b, int n, int P, float* __restrict__ bc, int Pc,
                                        float omega, const MgStrip& t, int lane) {
    constexpr int HALO = 3, H = MG_TY + 2 * HALO;
    float X[H], B[H];
    mg_load<H, EDGE>(B, b, t, n, P);
    if (p) {
        mg_load<H, EDGE>(X, p, t, n, P);
    } else {
#pragma unroll
        for (int q = 0; q < H; ++q) X[q] = 0.f;
    }
    mg_sweep<H, 1, EDGE>(X, B, t, n, omega);
    mg_sweep<H, 2, EDGE>(X, B, t, n, omega);
    const bool mine = lane >= 4 && lane < 4 + MG_TX && t.gj <= n;
#pragma unroll
    for (int q = HALO; q < HALO + MG_TY; q += 2) {
        float r[2];
#pragma unroll
        for (int d = 0; d < 2; ++d) {
            const int gi = t.gi0 + q + d;
            const float c = X[q + d];
            float nn = X[q + d - 1], ss = X[q + d + 1], ww = lane_west(c), ee = lane_east(c);
            if (EDGE) {
                nn = gi == 1 ? c : nn;
                ss = gi == n ? c : ss;
                ww = t.left ? c : ww;
                ee = t.right ? c : ee;
            }
            r[d] = B[q + d] - (4.f * c - nn - ss - ww - ee);
            if (mine && (!EDGE || gi <= n)) out[(size_t)gi * P + t.gj] = c;
        }
        const float r0e = lane_east(r[0]), r1e = lane_east(r[1]);
        if (mine && !(lane & 1) && (!EDGE || t.gi0 + q <= n)) {
            float sum = 0.f;
            sum += r[0];
            sum += r0e;
            sum += r[1];
            sum += r1e;
            bc[(size_t)((t.gi0 + q + 1) / 2) * Pc + (t.gj + 1) / 2] = sum;
        }
    }
}

// p plus the correction interpolated from pc, then two sweeps, into out (its ring too).
template <bool EDGE>
__device__ __forceinline__ void mg_up(const float* __restrict__ p, float* __restrict__ out, const float* __restrict__ b,
                                      int n, int P, const float* __restrict__ pc, int Pc, float omega,
                                      const MgStrip& t, int lane) {
    constexpr int HALO = 2, H = MG_TY + 2 * HALO, HC = H / 2 + 2;
    const int nc = n / 2;
    float X[H], B[H], C[HC], D[HC];
    mg_load<H, EDGE>(B, b, t, n, P);
    mg_load<H, EDGE>(X, p, t, n, P);
    // Fine cell i lies a quarter coarse cell from the centre of coarse cell
    // I = (i + 1) / 2, towards I0 = I - 1 (odd i) or I + 1; past the edge I0 is I.
    const int J = min(max((t.gj + 1) / 2, 1), nc), J0 = min(max((t.gj & 1) ? J - 1 : J + 1, 1), nc);
    const int k0 = (t.gi0 + 1) / 2 - 1;  // coarse row of C[0]; gi0 is odd
#pragma unroll
    for (int m = 0; m < HC; ++m) {
        const float* r = pc + (size_t)(EDGE ? min(max(k0 + m, 1), nc) : k0 + m) * Pc;
        C[m] = r[J];
        D[m] = r[J0];
    }
#pragma unroll
    for (int q = 0; q < H; ++q) {
        const int m = q / 2 + 1, m0 = (q & 1) ? m + 1 : m - 1;
        X[q] = X[q] + (0.5625f * C[m] + 0.1875f * D[m] + 0.1875f * C[m0] + 0.0625f * D[m0]);
    }
    mg_sweep<H, 1, EDGE>(X, B, t, n, omega);
    mg_sweep<H, 2, EDGE>(X, B, t, n, omega);
    if (lane < 4 || lane >= 4 + MG_TX || t.gj > n) return;
#pragma unroll
    for (int q = HALO; q < HALO + MG_TY; ++q) {
        const int gi = t.gi0 + q;
        if (!EDGE) out[(size_t)gi * P + t.gj] = X[q];
        else if (gi <= n) write_with_ring(out, gi, t.gj, n, P, X[q]);
    }
}

// The wave's tile; false where the block has more waves than tiles are left.
__device__ __forceinline__ bool mg_tile(int n, int halo, MgStrip& t, int& lane, bool& edge) {
    const int tiles_x = (n + MG_TX - 1) / MG_TX, tiles_y = (n + MG_TY - 1) / MG_TY, tiles = tiles_x * tiles_y;
    const int w = blockIdx.x * MG_WAVES + (threadIdx.x >> 6);
    if (w >= tiles) return false;
    lane = threadIdx.x & 63;
    t.gi0 = 1 + (w / tiles_x) * MG_TY - halo;
    const int gj0 = 1 + (w % tiles_x) * MG_TX - 4;
    t.gj = gj0 + lane;
    t.left = t.gj == 1;
    t.right = t.gj == n;
    edge = t.gi0 < 2 || t.gi0 + MG_TY + 2 * halo > n || gj0 < 2 || gj0 + 64 > n;
    return true;
}

__global__ __launch_bounds__(64 * MG_WAVES) void k_mg_down(const float* __restrict__ p, float* __restrict__ out,
                                                           const float* __restrict__ b, int n, int P,
                                                           float* __restrict__ bc, int Pc, float omega) {
    MgStrip t;
    int lane;
    bool edge;
    if (!mg_tile(n, 3, t, lane, edge)) return;
    if (edge) mg_down<true>(p, out, b, n, P, bc, Pc, omega, t, lane);
    else mg_down<false>(p, out, b, n, P, bc, Pc, omega, t, lane);
}

__global__ __launch_bounds__(64 * MG_WAVES) void k_mg_up(const float* __restrict__ p, float* __restrict__ out,
                                                         const float* __restrict__ b, int n, int P,
                                                         const float* __restrict__ pc, int Pc, float omega) {
    MgStrip t;
    int lane;
    bool edge;
    if (!mg_tile(n, 2, t, lane, edge)) return;
    if (edge) mg_up<true>(p, out, b, n, P, pc, Pc, omega, t, lane);
    else mg_up<false>(p, out, b, n, P, pc, Pc, omega, t, lane);
}

// ---- the tail: all levels of side n <= kMgTailSide in one block
constexpr int TAIL_THREADS = 1024, TAIL_WAVES = 16;
// iterates of sides 128, 64, 32, 16, 8 and 4, right-hand sides from 64 down
constexpr int TAIL_P = 16384 + 4096 + 1024 + 256 + 64 + 16, TAIL_B = TAIL_P - 16384;
constexpr int TAIL_EX = 2 * TAIL_WAVES * 2 * 128;  // the coarsest sweeps' row exchange

// `sweeps` sweeps of an n x n grid in LDS (p) with its right-hand side in the
// loader b: a wave holds RPW rows x 64 CPL columns in registers, neighbouring
// lanes exchange columns by DPP and neighbouring waves their edge rows
// through LDS, alternating between two buffers (one barrier a sweep).
template <int CPL, int RPW, class Rhs>
__device__ void tail_sweeps(float* __restrict__ p, const Rhs& b, int n, int sweeps, float omega, float* __restrict__ ex) {
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int i0 = wave * RPW, j0 = lane * CPL;
    float X[RPW][CPL], B[RPW][CPL];
#pragma unroll
    for (int r = 0; r < RPW; ++r)
#pragma unroll
        for (int c = 0; c < CPL; ++c) {
            const int i = min(i0 + r, n - 1), j = min(j0 + c, n - 1);
            X[r][c] = p[i * n + j];
            B[r][c] = b(i, j);
        }
    for (int s = 0; s < sweeps; ++s) {
        float* const e = ex + (s & 1) * TAIL_WAVES * 2 * 128;
#pragma unroll
        for (int c = 0; c < CPL; ++c) {
            e[(wave * 2) * 128 + j0 + c] = X[0][c];
            e[(wave * 2 + 1) * 128 + j0 + c] = X[RPW - 1][c];
        }
        __syncthreads();
        float above[CPL], below[CPL];
#pragma unroll
        for (int c = 0; c < CPL; ++c) {
            above[c] = CPL > 1 && wave == 0 ? X[0][c] : e[(max(wave - 1, 0) * 2 + 1) * 128 + j0 + c];
            below[c] = e[(min(wave + 1, TAIL_WAVES - 1) * 2) * 128 + j0 + c];
        }
#pragma unroll
        for (int r = 0; r < RPW; ++r) {
            float old[CPL];
#pragma unroll
            for (int c = 0; c < CPL; ++c) old[c] = X[r][c];
            // (two columns: lane 0, with no lane to its west, is given its own first
            // column by the shift; with one, the select below measured faster)
            const float west = CPL == 1 ? lane_west(old[CPL - 1])
                                        : __int_as_float(__builtin_amdgcn_update_dpp(
                                              __float_as_int(old[0]), __float_as_int(old[CPL - 1]), 0x138, 0xf, 0xf, false));
            const float east = lane_east(old[0]);
#pragma unroll
            for (int c = 0; c < CPL; ++c) {
                const float v = old[c];
                const float nn = CPL == 1 && i0 + r == 0 ? v : above[c];
                const float ss = i0 + r == n - 1 ? v : (r + 1 < RPW ? X[r + 1 < RPW ? r + 1 : r][c] : below[c]);
                const float ww = c > 0 ? old[c > 0 ? c - 1 : 0] : (CPL == 1 && j0 == 0 ? v : west);
                const float ee = j0 + c == n - 1 ? v : (c + 1 < CPL ? old[c + 1 < CPL ? c + 1 : c] : east);
                X[r][c] = smoothed(v, B[r][c], nn, ss, ww, ee, omega);
            }
#pragma unroll
            for (int c = 0; c < CPL; ++c) above[c] = old[c];
        }
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < RPW; ++r)
#pragma unroll
        for (int c = 0; c < CPL; ++c)
            if (i0 + r < n && j0 + c < n) p[(i0 + r) * n + j0 + c] = X[r][c];
    __syncthreads();
}

// The same for n * n <= 64: one wave, a cell a lane.
__device__ void tail_sweeps_small(float* __restrict__ p, const float* __restrict__ b, int n, int sweeps, float omega) {
    if (threadIdx.x < 64) {
        const int l = threadIdx.x, cells = n * n, q = min(l, cells - 1);
        const int i = q / n, j = q % n;
        const int ln = i == 0 ? q : q - n, ls = i == n - 1 ? q : q + n, lw = j == 0 ? q : q - 1, le = j == n - 1 ? q : q + 1;
        float v = p[q];
        const float bb = b[q];
        for (int s = 0; s < sweeps; ++s) {
            const float nn = __shfl(v, ln), ss = __shfl(v, ls), ww = __shfl(v, lw), ee = __shfl(v, le);
            v = smoothed(v, bb, nn, ss, ww, ee, omega);
        }
        if (l < cells) p[q] = v;
    }
    __syncthreads();
}

// A V-cycle from side n down: two sweeps, restriction, ..., `coarsest` sweeps
// of the last grid, ..., correction, two sweeps.  p is the level's iterate
// (pitch P; all zero where `zero`), b its right-hand side; `levels` grids in all.
__global__ __launch_bounds__(TAIL_THREADS) void k_mg_tail(float* __restrict__ p, const float* __restrict__ b, int n,
                                                          int P, int levels, int coarsest, int zero, float omega) {
    __shared__ float ps[TAIL_P], bs[TAIL_B], ex[TAIL_EX];
    const int tid = threadIdx.x;
    int np = n;
    float *pl = ps, *bl = bs;  // this level's; bl from the second level on
    // Two sweeps of a level: in registers for the wider grids; on those of at most
    // 16 x 16 cells on the LDS array itself, a cell a thread.
    auto smooth = [&](int side, float* x, const auto& rhs) {
        if (side > 64) return tail_sweeps<2, 8>(x, rhs, side, 2, omega, ex);
        if (side > 16) return tail_sweeps<1, 4>(x, rhs, side, 2, omega, ex);
        const int i = tid / side, j = tid % side, o = tid;
        const bool in = i < side;
        for (int sweep = 0; sweep < 2; ++sweep) {
            float v = 0.f;
            if (in) {
                const float c = x[o];
                v = smoothed(c, rhs(i, j), i == 0 ? c : x[o - side], i == side - 1 ? c : x[o + side],
                             j == 0 ? c : x[o - 1], j == side - 1 ? c : x[o + 1], omega);
            }
            __syncthreads();
            if (in) x[o] = v;
            __syncthreads();
        }
    };
    auto global_rhs = [&](int i, int j) { return b[(size_t)(i + 1) * P + j + 1]; };
    // down
    for (int q = tid; q < n * n; q += TAIL_THREADS) ps[q] = zero ? 0.f : p[(size_t)(q / n + 1) * P + q % n + 1];
    __syncthreads();
    for (int l = 0; l + 1 < levels; ++l) {
        const float* const cur = bl;
        auto lds_rhs = [&](int i, int j) { return cur[i * np + j]; };
        if (l == 0) smooth(np, pl, global_rhs);
        else smooth(np, pl, lds_rhs);
        const int nc = np / 2;
        float* const bn = l == 0 ? bs : bl + np * np;  // the next level's right-hand side
        float* const pn = pl + np * np;                // and iterate
        for (int q = tid; q < nc * nc; q += TAIL_THREADS) {
            const int I = q / nc, J = q % nc;
            float sum = 0.f;
#pragma unroll
            for (int di = 0; di < 2; ++di)
#pragma unroll
                for (int dj = 0; dj < 2; ++dj) {
                    const int i = 2 * I + di, j = 2 * J + dj, o = i * np + j;
                    const float c = pl[o];
                    const float nn = i == 0 ? c : pl[o - np], ss = i == np - 1 ? c : pl[o + np];
                    const float ww = j == 0 ? c : pl[o - 1], ee = j == np - 1 ? c : pl[o + 1];
                    sum += (l == 0 ? global_rhs(i, j) : lds_rhs(i, j)) - (4.f * c - nn - ss - ww - ee);
                }
            bn[q] = sum;
            pn[q] = 0.f;
        }
        __syncthreads();
        pl = pn;
        bl = bn;
        np = nc;
    }
    // coarsest
    {
        const float* const cur = bl;
        auto lds_rhs = [&](int i, int j) { return cur[i * np + j]; };
        if (levels == 1) {
            if (np <= 64) tail_sweeps<1, 4>(pl, global_rhs, np, coarsest, omega, ex);
            else tail_sweeps<2, 8>(pl, global_rhs, np, coarsest, omega, ex);
        } else if (np * np <= 64) {
            tail_sweeps_small(pl, cur, np, coarsest, omega);
        } else {
            tail_sweeps<1, 4>(pl, lds_rhs, np, coarsest, omega, ex);  // a second level's side is at most 64
        }
    }
    // up
    for (int l = levels - 2; l >= 0; --l) {
        const int nc = np, nf = 2 * nc;
        const float* const pc = pl;
        pl -= nf * nf;
        if (l > 0) bl -= nf * nf;
        np = nf;
        for (int q = tid; q < nf * nf; q += TAIL_THREADS) {
            const int i = q / nf + 1, j = q % nf + 1;
            const int I = (i + 1) / 2, J = (j + 1) / 2;
            const int I0 = min(max((i & 1) ? I - 1 : I + 1, 1), nc), J0 = min(max((j & 1) ? J - 1 : J + 1, 1), nc);
            pl[q] += 0.5625f * pc[(I - 1) * nc + J - 1] + 0.1875f * pc[(I - 1) * nc + J0 - 1] +
                     0.1875f * pc[(I0 - 1) * nc + J - 1] + 0.0625f * pc[(I0 - 1) * nc + J0 - 1];
        }
        __syncthreads();
        const float* const cur = bl;
        auto lds_rhs = [&](int i, int j) { return cur[i * np + j]; };
        if (l == 0) smooth(np, pl, global_rhs);
        else smooth(np, pl, lds_rhs);
    }
    for (int q = tid; q < n * n; q += TAIL_THREADS) write_with_ring(p, q / n + 1, q % n + 1, n, P, ps[q]);
}

dim3 interior_grid(int n) { return dim3((n + kMgThreads - 1) / kMgThreads, n); }

dim3 tile_grid(int n) {
    const int tiles = ((n + MG_TX - 1) / MG_TX) * ((n + MG_TY - 1) / MG_TY);
    return dim3((tiles + MG_WAVES - 1) / MG_WAVES);
}

}  // namespace

hipError_t launch_mg_smooth(hipStream_t s, const float* src, float* dst, const float* b, int R, int P, float omega) {
    hipLaunchKernelGGL(k_mg_smooth, interior_grid(R - 2), dim3(kMgThreads), 0, s, src, dst, b, R, P, omega);
    return hipGetLastError();
}

hipError_t launch_mg_down(hipStream_t s, const float* p, float* out, const float* b, int n, int P, float* bc, int Pc,
                          float omega) {
    hipLaunchKernelGGL(k_mg_down, tile_grid(n), dim3(64 * MG_WAVES), 0, s, p, out, b, n, P, bc, Pc, omega);
    return hipGetLastError();
}

hipError_t launch_mg_up(hipStream_t s, const float* p, float* out, const float* b, int n, int P, const float* pc,
                        int Pc, float omega) {
    hipLaunchKernelGGL(k_mg_up, tile_grid(n), dim3(64 * MG_WAVES), 0, s, p, out, b, n, P, pc, Pc, omega);
    return hipGetLastError();
}

hipError_t launch_mg_tail(hipStream_t s, float* p, const float* b, int n, int P, int levels, int coarsest, bool zero,
                          float omega) {
    hipLaunchKernelGGL(k_mg_tail, dim3(1), dim3(TAIL_THREADS), 0, s, p, b, n, P, levels, coarsest, zero ? 1 : 0, omega);
    return hipGetLastError();
}

}  // namespace fs2d
