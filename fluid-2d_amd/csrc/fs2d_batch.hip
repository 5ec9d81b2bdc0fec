// fs2d_batch.hip -- many independent simulations of different sizes, one
// launch per stage (declared in include/fs2d_hip.h, fs2d_hip_batch_*).
//
// Layout: every field kind (density, u, v, the sources, the diffuse and
// pressure iterates and right-hand sides, the Jacobi scratch pairs) is one
// arena holding all simulations' grids; simulation s occupies the same range
// [off_s, off_s + R_s * P_s) in every arena, with its own row pitch P_s (R_s
// rounded up to 64 floats).  Swapping two arenas therefore swaps that role
// for every simulation at once, so the buffer rotation of the step stays a
// host-side permutation of arena pointers, identical for all simulations.
//
// Each stage is one launch over a work list: the single-pass stages over
// (simulation, 64 x 4 cell block) entries, the Jacobi sweeps over
// (simulation, field, tile) entries with the block tile of the one-grid solver, or, in
// fixed launches of one or two sweeps, over (simulation, field, strip) entries.
// Simulation s runs its K_s sweeps in L_s launches of at most 8 fused sweeps,
// as evenly as they go; launch j covers the simulations with more than j
// launches (the work list is ordered by launch count, so that is a prefix of
// it), and ping-pongs home -> S1 -> S2 -> S1 ... -> home, so that every solve
// ends in its home field whatever its launch count (L_s >= 2).
//
// The step follows fluid_solver_cpu::solve (src/fluid_solver_cpu.cpp:6-31)
// in the Jacobi order, exactly as fs2d_handle's step does: each simulation's
// fields come out bit-identical to a one-grid handle with the same inputs.
#include "../../include/fs2d_hip.h"
#include "fs2d_cells.hpp"
#include "fs2d_internal.hpp"
#include "fs2d_jacobi.hpp"

#include <algorithm>
#include <cmath>
#include <cstring>
#include <exception>
#include <new>
#include <string>
#include <vector>

using namespace fs2d;

namespace {

thread_local std::string g_batch_create_error;

// Arena roles.  The diffuse solves of density, u and v use (home, rhs,
// scratch pair) = (RHO, X0, S1A/S2A), (UN, X0U, S1B/S2B), (VN, X0V, S1C/S2C);
// the pressure solve uses (P, D, S1A/S2A).
enum {
    A_RHO, A_U, A_V, A_RS, A_US, A_VS, A_X0, A_X0U, A_X0V, A_UN, A_VN, A_T1, A_T2, A_D, A_P,
    A_S1A, A_S2A, A_S1B, A_S2B, A_S1C, A_S2C, A_COUNT
};

struct Roles {
    float* a[A_COUNT];
};

// Per-simulation constants, computed on the host exactly as the one-grid
// handle computes them.
struct BatchSim {
    size_t off;  // floats, 256-byte aligned
    int R, P;
    int launches;     // Jacobi launches per solve (diffuse and pressure)
    int sweeps;       // fewest sweeps of a launch; the first `longer` launches have one more
    int longer;
    float dt, dt0, h, neg_half_h;
    float a_rho, a_vel;
    jac::Divisor dv_rho, dv_vel;
    int checked_rho, checked_vel;  // the divisor has a known quotient (known_quotient)
};

constexpr int CBX = 64, CBY = 4;      // single-pass stage blocks
constexpr int kSimSlots = 16;         // speed-reduction slots per simulation
constexpr int kSimSlotStride = 32;    // words between slots (separate cache lines)

__device__ __forceinline__ int xcd_block(int b, int nb) { return jac::xcd_block(b, nb); }

// Single-pass stages are persistent: block b walks entries b, b + G, ... of
// the work list (G blocks, a multiple of 8: each block's entries then map,
// through xcd_block, into one contiguous run of the list per XCD).
// Entry e: x = simulation, y = (by << 16) | bx.
__device__ __forceinline__ bool cell_of(const BatchSim* __restrict__ sims, const int2* __restrict__ work, int e,
                                        int nb, int& s, int& i, int& j, int& blk) {
    const int2 w = work[xcd_block(e, nb)];
    s = w.x;
    const int bx = w.y & 0xffff, by = w.y >> 16;
    j = bx * CBX + threadIdx.x + 1;
    i = by * CBY + threadIdx.y + 1;
    blk = w.y;
    const int R = sims[s].R;
    return i <= R - 2 && j <= R - 2;
}

// Block maximum of the largest finite |u|, |v| into one of the simulation's
// slots (k_fold folds them).  Ends with a barrier, so a persistent block may
// reduce its next entry at once.
__device__ __forceinline__ void speed_to_slot(float m, unsigned* __restrict__ slots, int s, int blk) {
    m = cells::block_max(m);
    if (threadIdx.x == 0 && threadIdx.y == 0) {
        const unsigned slot = (unsigned)((blk & 0xffff) + 131 * (blk >> 16)) % kSimSlots;
        atomicMax(slots + ((size_t)s * kSimSlots + slot) * kSimSlotStride, __float_as_uint(m));
    }
    __syncthreads();
}

__global__ __launch_bounds__(CBX* CBY) void kb_max_speed(const BatchSim* __restrict__ sims,
                                                         const int2* __restrict__ work, int nwork, Roles r,
                                                         unsigned* __restrict__ slots) {
    for (int e = blockIdx.x; e < nwork; e += gridDim.x) {
        int s, i, j, blk;
        const bool in = cell_of(sims, work, e, nwork, s, i, j, blk);
        float m = 0.f;
        if (in) {
            const size_t o = sims[s].off + (size_t)i * sims[s].P + j;
            m = cells::fold_speed(0.f, r.a[A_U][o], r.a[A_V][o]);
        }
        speed_to_slot(m, slots, s, blk);
    }
}

// One 64-lane block per simulation: fold its slots into max_bits[s] and clear them.
__global__ __launch_bounds__(64) void kb_fold_speed(unsigned* __restrict__ max_bits, unsigned* __restrict__ slots) {
    const int s = blockIdx.x, t = threadIdx.x;
    unsigned m = 0u;
    if (t < kSimSlots) {
        unsigned* p = slots + ((size_t)s * kSimSlots + t) * kSimSlotStride;
        m = *p;
        *p = 0u;
    }
    for (int off = 32; off > 0; off >>= 1) m = max(m, (unsigned)__shfl_xor((int)m, off));
    if (t == 0) max_bits[s] = m;
}

__global__ __launch_bounds__(CBX* CBY) void kb_gather_velocity(const BatchSim* __restrict__ sims,
                                                               const int2* __restrict__ work, int nwork, Roles r) {
    for (int e = blockIdx.x; e < nwork; e += gridDim.x) {
        int s, i, j, blk;
        if (!cell_of(sims, work, e, nwork, s, i, j, blk)) continue;
        const BatchSim& S = sims[s];
        const size_t o = S.off;
        cells::gather_velocity(r.a[A_T1] + o, r.a[A_T2] + o, r.a[A_U] + o, r.a[A_V] + o, S.R, S.P, S.dt0, i, j);
    }
}

__global__ __launch_bounds__(CBX* CBY) void kb_gradient(const BatchSim* __restrict__ sims,
                                                        const int2* __restrict__ work, int nwork, Roles r,
                                                        unsigned* __restrict__ slots) {
    for (int e = blockIdx.x; e < nwork; e += gridDim.x) {
        int s, i, j, blk;
        const bool in = cell_of(sims, work, e, nwork, s, i, j, blk);
        float m = 0.f;
        if (in) {
            const BatchSim& S = sims[s];
            const size_t o = S.off;
            m = cells::gradient(r.a[A_U] + o, r.a[A_V] + o, r.a[A_P] + o, S.R, S.P, S.h, false, i, j);
        }
        if (slots) speed_to_slot(m, slots, s, blk);
    }
}

// Jacobi launch j over (simulation, field, tile) entries: x = simulation |
// field << 24, y = tile (row-major over tiles_y x tiles_x).  Persistent: block g
// of G takes entries g, g + G, ... (through xcd_block), each one block tile
// (fs2d_jacobi.hpp) of RPW JB_WAVES rows x 64 columns.
//
// What bounds it: VALU issue (a tile's halo of 8 rows and columns is 0.8 of a grid's
// cells at side 512, more on smaller ones) and memory, both at about half of a
// launch's time.  256 simulations of sides 64 to 512 (19.3 M cells, 20 or 40 sweeps),
// one step's diffuse solves / one pressure solve: one wave per 16-row tile, 4 sweeps
// a launch 1.50 / 0.45 ms; block tiles of 48 rows, at most 8 sweeps a launch 1.41 /
// 0.40 ms; of 96 rows 1.21 / 0.38 ms; with known ring rows and lanes, and the right-hand
// sides formed by the first launches, 1.12 / 0.33 ms (the sources' pass of 0.25 ms and a
// divergence's 0.06 ms are in these and were not before).  The gradient stays a pass:
// made by the last launch, 40 steps and their read-back took 106.0 ms against 101.9.
constexpr int JB_WAVES = 8;

// Launch j's job of one field: what it reads and writes, and the divisor; whether that
// is a checked one.
template <int KIND, bool FIRST>
__device__ __forceinline__ bool batch_job(const BatchSim& S, const Roles& r, int f, int j, jac::TileJob& t) {
    const size_t o = S.off;
    t.R = S.R;
    t.P = S.P;
    bool checked = false;
    float *home, *s1, *s2;
    if (KIND == SWEEP_PRESSURE) {
        home = r.a[A_P] + o;
        t.b = r.a[A_D] + o;
        s1 = r.a[A_S1A] + o;
        s2 = r.a[A_S2A] + o;
        t.rg = ring_of(BND_CONT);
        t.a = 0.f;
        t.dv = jac::Divisor{};
        t.s0 = r.a[A_U] + o;
        t.s1 = r.a[A_V] + o;
        t.scale = S.neg_half_h;
        t.b_out = r.a[A_D] + o;
    } else {
        home = r.a[f == 0 ? A_RHO : (f == 1 ? A_UN : A_VN)] + o;
        t.b = r.a[f == 0 ? A_X0 : (f == 1 ? A_X0U : A_X0V)] + o;
        s1 = r.a[f == 0 ? A_S1A : (f == 1 ? A_S1B : A_S1C)] + o;
        s2 = r.a[f == 0 ? A_S2A : (f == 1 ? A_S2B : A_S2C)] + o;
        t.rg = ring_of(f == 0 ? BND_CONT : (f == 1 ? BND_OPP_H : BND_OPP_V));
        t.a = f == 0 ? S.a_rho : S.a_vel;
        t.dv = f == 0 ? S.dv_rho : S.dv_vel;
        checked = (f == 0 ? S.checked_rho : S.checked_vel) != 0;
        // u and v go to fresh iterates: the density scatter reads the pre-step
        // velocity (:16-24)
        t.src = r.a[f == 0 ? A_RHO : (f == 1 ? A_U : A_V)] + o;
        t.s0 = r.a[f == 0 ? A_RS : (f == 1 ? A_US : A_VS)] + o;
        t.scale = S.dt;
        t.b_out = r.a[f == 0 ? A_X0 : (f == 1 ? A_X0U : A_X0V)] + o;
    }
    if (!FIRST) t.src = ((j - 1) & 1) ? s2 : s1;
    t.dst = (j == S.launches - 1) ? home : ((j & 1) ? s2 : s1);
    t.zero = false;
    return checked;
}

// A solve's first launch (FIRST, j = 0) forms its right-hand sides: the sources' terms
// of density, u and v, or the divergence.
template <int RPW, int KIND, bool FIRST>
__global__ __launch_bounds__(64 * JB_WAVES) void kb_jacobi(const BatchSim* __restrict__ sims,
                                                           const int2* __restrict__ work, int n_work, Roles r,
                                                           int j) {
    __shared__ float ex[4 * JB_WAVES * jac::kTileCols];
    for (int e = xcd_block(blockIdx.x, gridDim.x); e < n_work; e += gridDim.x) {
        const int2 w = work[e];
        const int s = w.x & 0xffffff, f = w.x >> 24;
        const BatchSim& S = sims[s];
        jac::TileJob t;
        const bool checked = batch_job<KIND, FIRST>(S, r, f, j, t);
        // tiles are placed for the longest launch
        t.m = S.sweeps + (S.longer > 0);
        const int tiles_y = jac::tile_count(t.R, RPW * JB_WAVES, t.m), tiles_x = jac::tile_count(t.R, jac::kTileCols, t.m);
        const int ty = w.y / tiles_x;
        jac::tile_place(t, RPW * JB_WAVES, ty, w.y - ty * tiles_x, tiles_y, tiles_x);
        t.m = S.sweeps + (j < S.longer);
        if constexpr (KIND == SWEEP_PRESSURE)
            jac::jacobi_tile_any<RPW, JB_WAVES, jac::TILE_PRESSURE, FIRST ? jac::TILE_DIVERGENCE : jac::TILE_STORED>(t, ex);
        else if (checked)
            jac::jacobi_tile_any<RPW, JB_WAVES, jac::TILE_DIFFUSE_CHECKED, FIRST ? jac::TILE_SOURCES : jac::TILE_STORED>(t, ex);
        else
            jac::jacobi_tile_any<RPW, JB_WAVES, jac::TILE_DIFFUSE, FIRST ? jac::TILE_SOURCES : jac::TILE_STORED>(t, ex);
        __syncthreads();  // the next tile's first exchange may take the buffer of this one's last
    }
}

// A launch of M = 1 or 2 sweeps that is not a solve's first, one wave a strip: lane l
// holds column gj0 + l of a 64-column region and its kStripRows + 2M rows in registers.
// Each sweep leaves one more row and lane a side stale; rows M .. and lanes M .. 63 - M
// are written.  Region cells outside the grid hold clamped values that reach only other
// outside cells or the ring, which is rebuilt from the new interior after a sweep.
//
// What bounds it: memory, at one or two sweeps a pass.  A block tile's waves wait for
// each other each sweep and its rows past the grid's are relaxed in vain, which so few
// sweeps do not pay back.  A step by tiles and by strips, us: 300 grids of 66 x 66, 20
// sweeps, 1 a launch 1099 and 711, 2 a launch 632 and 511; 512 of 98 x 98, 16 sweeps,
// 1940 and 1349, 1166 and 934; 256 of sides 64 to 512 9292 and 8669, 5007 and 4846; one
// of 4098 x 4098 4277 and 4065, 2430 and 2419.  From 4 sweeps a launch on tiles win
// (256 grids: 2941 us).  Strips of 32 rows take the same time.
constexpr int kStripRows = 16, kStripWaves = 4;

__host__ __device__ inline int strip_count(int R, int m) {
    const int n = R - 2, cols = 64 - 2 * m;
    return ((n + cols - 1) / cols) * ((n + kStripRows - 1) / kStripRows);
}

template <int M, int KIND, bool EDGE>
__device__ __forceinline__ void batch_strip(const jac::TileJob& t, int gi0, int gj0, int lane) {
    constexpr int H = kStripRows + 2 * M;
    const int R = t.R, P = t.P, n = R - 2, gj = gj0 + lane;
    float X[H], B[H];
    if (EDGE) {
        const int cj = min(max(gj, 0), R - 1), bj = min(max(gj, 1), n);
#pragma unroll
        for (int q = 0; q < H; ++q) X[q] = t.src[(size_t)min(max(gi0 + q, 0), R - 1) * P + cj];
#pragma unroll
        for (int q = 1; q < H - 1; ++q) B[q] = t.b[(size_t)min(max(gi0 + q, 1), n) * P + bj];
    } else {
        const size_t o = (size_t)gi0 * P + gj;
#pragma unroll
        for (int q = 0; q < H; ++q) X[q] = t.src[o + (size_t)q * P];
#pragma unroll
        for (int q = 1; q < H - 1; ++q) B[q] = t.b[o + (size_t)q * P];
    }
    const bool cols_ring = EDGE && (gj0 <= 0 || gj0 + 63 >= R - 1);  // the same in all lanes
#pragma unroll
    for (int s = 1; s <= M; ++s) {
        float north = X[s - 1];
#pragma unroll
        for (int q = s; q < H - s; ++q) {
            const float c = X[q];
            float v = jac::relax_k<KIND>(B[q], north, X[q + 1], jac::lane_west(c), jac::lane_east(c), t.a, t.dv);
            north = c;
            if (EDGE && s < M) {
                const int gi = gi0 + q;
                if (gi == R - 1) v = jac::sgn(t.rg.neg_tb, X[q - 1]);
                if (cols_ring) {
                    const float e = jac::sgn(t.rg.neg_lr, jac::lane_east(v)), w = jac::sgn(t.rg.neg_lr, jac::lane_west(v));
                    v = gj == 0 ? e : (gj == R - 1 ? w : v);
                }
                if (gi == 1) X[q - 1] = jac::sgn(t.rg.neg_tb, v);
            }
            X[q] = v;
        }
    }
    if (lane < M || lane >= 64 - M || gj > n) return;  // gj >= 1: a strip starts at column 1 - M
#pragma unroll
    for (int q = M; q < M + kStripRows; ++q) {
        const int gi = gi0 + q;
        if (EDGE && gi > n) continue;
        t.dst[(size_t)gi * P + gj] = X[q];
        if (EDGE) cells::write_ring(t.dst, gi, gj, X[q], R, P, t.rg);
    }
}

// Entries as kb_jacobi's, the strips of a field row-major.  LOOP: persistent by waves,
// else an entry a wave (the loop's code cost launches of one sweep 5 %).
template <int M, int KIND, bool LOOP>
__global__ __launch_bounds__(64 * kStripWaves) void kb_strip(const BatchSim* __restrict__ sims,
                                                             const int2* __restrict__ work, int n_work, Roles r, int j) {
    const int lane = threadIdx.x & 63, waves = (int)gridDim.x * kStripWaves;
    // (no barrier: a wave leaves when its entries are done)
    for (int e = xcd_block(blockIdx.x, gridDim.x) * kStripWaves + (threadIdx.x >> 6); e < n_work; e += waves) {
        const int2 w = work[e];
        const BatchSim& S = sims[w.x & 0xffffff];
        jac::TileJob t;
        batch_job<KIND, false>(S, r, w.x >> 24, j, t);
        constexpr int cols = 64 - 2 * M;
        const int across = (t.R - 2 + cols - 1) / cols, ty = w.y / across;
        const int gi0 = 1 + kStripRows * ty - M, gj0 = 1 + cols * (w.y - ty * across) - M;
        const bool plain = gi0 >= 1 && gi0 + kStripRows + 2 * M - 1 <= t.R - 2 && gj0 >= 1 && gj0 + 63 <= t.R - 2;
        if (plain) batch_strip<M, KIND, false>(t, gi0, gj0, lane);
        else batch_strip<M, KIND, true>(t, gi0, gj0, lane);
        if (!LOOP) return;
    }
}

__global__ __launch_bounds__(256) void kb_fill(uint32_t* __restrict__ p, size_t n) {
    for (size_t t = (size_t)blockIdx.x * 256 + threadIdx.x; t < n; t += (size_t)gridDim.x * 256) p[t] = 0u;
}

// Blocks of a persistent launch over `n` entries of `per_block` each, at most
// `limit` (a multiple of 8 when it binds, so that every block's entries fall
// in one XCD's run of the list).
unsigned persistent_grid(int n, int per_block, int limit) {
    const int need = (n + per_block - 1) / per_block;
    if (limit <= 0 || need <= limit) return static_cast<unsigned>(std::max(need, 1));
    return static_cast<unsigned>(std::max(8, limit - limit % 8));
}

template <int RPW, int KIND>
void launch_kb_jacobi_kind(hipStream_t st, const BatchSim* sims, const int2* w, int n, Roles r, int j, int limit) {
    const dim3 grid(persistent_grid(n, 1, limit)), block(64 * JB_WAVES);
    if (j == 0) hipLaunchKernelGGL((kb_jacobi<RPW, KIND, true>), grid, block, 0, st, sims, w, n, r, j);
    else hipLaunchKernelGGL((kb_jacobi<RPW, KIND, false>), grid, block, 0, st, sims, w, n, r, j);
}

template <int RPW>
void launch_kb_jacobi_rows(hipStream_t st, int kind, const BatchSim* sims, const int2* w, int n, Roles r, int j,
                           int limit) {
    if (kind == SWEEP_DIFFUSE) launch_kb_jacobi_kind<RPW, SWEEP_DIFFUSE>(st, sims, w, n, r, j, limit);
    else launch_kb_jacobi_kind<RPW, SWEEP_PRESSURE>(st, sims, w, n, r, j, limit);
}

hipError_t launch_kb_jacobi(hipStream_t st, int rows, int kind, const BatchSim* sims, const int2* w, int n, Roles r,
                            int j, int limit) {
    if (n <= 0) return hipSuccess;
    switch (rows) {
        case 32: launch_kb_jacobi_rows<4>(st, kind, sims, w, n, r, j, limit); break;
        case 48: launch_kb_jacobi_rows<6>(st, kind, sims, w, n, r, j, limit); break;
        case 96: launch_kb_jacobi_rows<12>(st, kind, sims, w, n, r, j, limit); break;
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

template <int M, int KIND>
void launch_kb_strip_kind(hipStream_t st, const BatchSim* sims, const int2* w, int n, Roles r, int j, int limit) {
    const dim3 grid(persistent_grid(n, kStripWaves, limit)), block(64 * kStripWaves);
    if (limit > 0) hipLaunchKernelGGL((kb_strip<M, KIND, true>), grid, block, 0, st, sims, w, n, r, j);
    else hipLaunchKernelGGL((kb_strip<M, KIND, false>), grid, block, 0, st, sims, w, n, r, j);
}

template <int M>
hipError_t launch_kb_strip(hipStream_t st, int kind, const BatchSim* sims, const int2* w, int n, Roles r, int j,
                           int limit) {
    if (n <= 0) return hipSuccess;
    if (kind == SWEEP_DIFFUSE) launch_kb_strip_kind<M, SWEEP_DIFFUSE>(st, sims, w, n, r, j, limit);
    else launch_kb_strip_kind<M, SWEEP_PRESSURE>(st, sims, w, n, r, j, limit);
    return hipGetLastError();
}

}  // namespace

// The work lists of the diffuse (3 fields) and pressure (1 field) solves with,
// for each launch j, the number of leading entries whose simulation runs launch j.
struct JacobiWork {
    int rows = 0;  // of a tile's region
    int2* diffuse = nullptr;
    int2* pressure = nullptr;
    std::vector<int> diffuse_count, pressure_count;  // per launch j
    // the same for the launches after a solve's first where they take strips
    int strip_sweeps = 0;  // 0: they take tiles
    int2* diffuse_strips = nullptr;
    int2* pressure_strips = nullptr;
    std::vector<int> diffuse_strip_count, pressure_strip_count;
};

struct BatchGraph {
    float* pre[A_COUNT];
    float* post[A_COUNT];
    bool pre_speed;
    hipGraph_t graph = nullptr;  // kept while its executable lives (tools inspect it at launch)
    hipGraphExec_t exec = nullptr;
};

struct fs2d_batch {
    int count = 0;
    fs2d_params prm{};
    std::vector<BatchSim> host_sims;
    std::vector<int> order;           // simulations by Jacobi launch count, descending
    size_t arena_floats = 0;
    long long interior = 0;
    hipStream_t stream = nullptr;
    HostStage stage;  // host transfers (fs2d_transfer.hip)
    Roles roles{};
    BatchSim* sims = nullptr;     // device copy of host_sims
    int2* cell_work = nullptr;    // single-pass stage blocks, all simulations
    int cell_blocks = 0;
    unsigned* max_bits = nullptr;  // per simulation
    unsigned* slots = nullptr;     // per simulation kSimSlots * kSimSlotStride words, zero between uses
    ScatterSim* scatter_sims = nullptr;  // the density scatter's descriptors (fs2d_scatter.hip)
    int2* scatter_windows = nullptr;     // its window path's work list, one entry per wave
    void* scatter_scratch = nullptr;     // its sorted path's buffers
    int* scatter_flag = nullptr;         // its sorted-path gate
    BatchScatter scatter{};
    int cus = 256;                // compute units of the device
    int jac_per_cu = 0;           // persistent Jacobi blocks per CU (0: one per entry)
    int cell_per_cu = 8;          // persistent single-pass blocks per CU (0: one per entry)
    JacobiWork jacobi;
    bool speed_valid = false;
    long long steps_done = 0;
    std::vector<BatchGraph*> graphs;
    std::string err;
};

namespace {

int bfail(fs2d_batch* b, int code, const std::string& msg) {
    if (b) b->err = msg;
    else g_batch_create_error = msg;
    return code;
}

#define FS2D_BHIP(b, expr)                                                                     \
    do {                                                                                       \
        hipError_t e_ = (expr);                                                                \
        if (e_ != hipSuccess)                                                                  \
            return bfail((b), FS2D_ERR_HIP, std::string(#expr) + ": " + hipGetErrorString(e_)); \
    } while (0)

float cells_of(int R) { return static_cast<float>(static_cast<size_t>(R) * static_cast<size_t>(R)); }

int jac_limit(const fs2d_batch* b) { return b->jac_per_cu > 0 ? b->cus * b->jac_per_cu : 0; }
dim3 cell_grid(const fs2d_batch* b) { return dim3(persistent_grid(b->cell_blocks, 1, b->cell_per_cu > 0 ? b->cus * b->cell_per_cu : 0)); }

// One solve kind's work list (`fields` fields a simulation, tiles(S) entries a field),
// and the prefix of it that launch j takes: entries are ordered by the simulation's
// launch count (descending).
template <class F>
hipError_t build_work(const fs2d_batch* b, int fields, F&& tiles, int2** list, std::vector<int>* counts) {
    std::vector<int2> w;
    for (int s : b->order) {
        const BatchSim& S = b->host_sims[s];
        const int n = tiles(S);
        for (int f = 0; f < fields; ++f)
            for (int t = 0; t < n; ++t) w.push_back(make_int2(s | (f << 24), t));
        if (counts->empty()) counts->assign(S.launches, 0);  // the first has the most launches
        for (int j = 0; j < S.launches; ++j) (*counts)[j] += fields * n;
    }
    const hipError_t e = hipMalloc(list, sizeof(int2) * w.size());
    return e != hipSuccess ? e : hipMemcpy(*list, w.data(), sizeof(int2) * w.size(), hipMemcpyHostToDevice);
}

// Tiles of one field of a simulation whose regions are `rows` high.
int tiles_of(const BatchSim& S, int rows) {
    const int m = S.sweeps + (S.longer > 0);
    return jac::tile_count(S.R, rows, m) * jac::tile_count(S.R, jac::kTileCols, m);
}

// Rows of a tile's region: as for one grid (fs2d_jacobi.hip), by the cells of a diffuse
// launch.  But many grids a little over one region high leave most of their second tile
// of 96 rows to the first: where regions of 48 rows hold less than 0.85 of the rows those
// of 96 do, they are the faster ones.  512 grids of 98 x 98, 16 sweeps, a step with 48
// and 96 rows (0.75): 554 and 619 us; at equal rows 400 of 130 x 130 961 and 886, 50 of
// 258 x 258 406 and 357, 700 of 66 x 66 604 and 628 us.
int jacobi_rows(const fs2d_batch* b) {
    const long long cells = 3 * b->interior;
    if (cells < 500000) return 32;
    if (cells < 8000000) return 48;
    double low = 0, high = 0;  // rows of regions relaxed in a solve
    for (const BatchSim& S : b->host_sims) {
        const double sweeps = static_cast<double>(S.launches) * S.sweeps + S.longer;
        low += sweeps * tiles_of(S, 48) * 48;
        high += sweeps * tiles_of(S, 96) * 96;
    }
    return low < 0.85 * high ? 48 : 96;
}

// Work lists of the Jacobi launches.  Fixed launches of 1 or 2 sweeps take strips after
// a solve's first one.
hipError_t build_jacobi_work(fs2d_batch* b) {
    JacobiWork& c = b->jacobi;
    c.rows = jacobi_rows(b);
    const auto tiles = [&](const BatchSim& S) { return tiles_of(S, c.rows); };
    hipError_t e;
    if ((e = build_work(b, 3, tiles, &c.diffuse, &c.diffuse_count)) != hipSuccess) return e;
    if ((e = build_work(b, 1, tiles, &c.pressure, &c.pressure_count)) != hipSuccess) return e;
    const int m = b->prm.jacobi_block;
    if (m != 1 && m != 2) return hipSuccess;
    c.strip_sweeps = m;
    const auto strips = [&](const BatchSim& S) { return strip_count(S.R, m); };
    if ((e = build_work(b, 3, strips, &c.diffuse_strips, &c.diffuse_strip_count)) != hipSuccess) return e;
    return build_work(b, 1, strips, &c.pressure_strips, &c.pressure_strip_count);
}

int solve(fs2d_batch* b, int kind) {
    const JacobiWork& c = b->jacobi;
    const bool diffuse = kind == SWEEP_DIFFUSE;
    const auto& counts = diffuse ? c.diffuse_count : c.pressure_count;
    const auto& strips = diffuse ? c.diffuse_strip_count : c.pressure_strip_count;
    const int2* w = diffuse ? c.diffuse : c.pressure;
    const int2* ws = diffuse ? c.diffuse_strips : c.pressure_strips;
    for (int j = 0; j < static_cast<int>(counts.size()); ++j) {
        if (j == 0 || !c.strip_sweeps)
            FS2D_BHIP(b, launch_kb_jacobi(b->stream, c.rows, kind, b->sims, w, counts[j], b->roles, j, jac_limit(b)));
        else if (c.strip_sweeps == 1)
            FS2D_BHIP(b, launch_kb_strip<1>(b->stream, kind, b->sims, ws, strips[j], b->roles, j, jac_limit(b)));
        else
            FS2D_BHIP(b, launch_kb_strip<2>(b->stream, kind, b->sims, ws, strips[j], b->roles, j, jac_limit(b)));
    }
    return FS2D_OK;
}

hipError_t cell_launch_check() { return hipGetLastError(); }

// speed: the largest speeds of the result are wanted too.
int project(fs2d_batch* b, bool speed) {
    const dim3 grid = cell_grid(b), blk(CBX, CBY);
    int rc = solve(b, SWEEP_PRESSURE);
    if (rc) return rc;
    hipLaunchKernelGGL(kb_gradient, grid, blk, 0, b->stream, b->sims, b->cell_work, b->cell_blocks, b->roles,
                       speed ? b->slots : nullptr);
    if (speed)
        hipLaunchKernelGGL(kb_fold_speed, dim3(b->count), dim3(64), 0, b->stream, b->max_bits, b->slots);
    FS2D_BHIP(b, cell_launch_check());
    return FS2D_OK;
}

// One step of every simulation (fluid_solver_cpu::solve, Jacobi order).
int step(fs2d_batch* b) {
    const dim3 blk(CBX, CBY);
    int rc;
    if (!b->speed_valid) {
        hipLaunchKernelGGL(kb_max_speed, cell_grid(b), blk, 0, b->stream, b->sims, b->cell_work, b->cell_blocks,
                           b->roles, b->slots);
        hipLaunchKernelGGL(kb_fold_speed, dim3(b->count), dim3(64), 0, b->stream, b->max_bits, b->slots);
        FS2D_BHIP(b, cell_launch_check());
        b->speed_valid = true;
    }
    if ((rc = solve(b, SWEEP_DIFFUSE))) return rc;
    FS2D_BHIP(b, launch_batch_scatter(b->stream, b->scatter, b->roles.a[A_T1], b->roles.a[A_RHO], b->roles.a[A_U],
                                      b->roles.a[A_V], b->max_bits));
    std::swap(b->roles.a[A_RHO], b->roles.a[A_T1]);
    std::swap(b->roles.a[A_U], b->roles.a[A_UN]);
    std::swap(b->roles.a[A_V], b->roles.a[A_VN]);
    if ((rc = project(b, false))) return rc;
    hipLaunchKernelGGL(kb_gather_velocity, cell_grid(b), blk, 0, b->stream, b->sims, b->cell_work, b->cell_blocks,
                       b->roles);
    FS2D_BHIP(b, cell_launch_check());
    std::swap(b->roles.a[A_U], b->roles.a[A_T1]);
    std::swap(b->roles.a[A_V], b->roles.a[A_T2]);
    return project(b, true);
}

constexpr size_t kMaxBatchGraphs = 16;

void drop_graphs(fs2d_batch* b) {
    for (auto* g : b->graphs) {
        if (g->exec) (void)hipGraphExecDestroy(g->exec);
        if (g->graph) (void)hipGraphDestroy(g->graph);
        delete g;
    }
    b->graphs.clear();
}

// As fs2d_handle's step graphs: the first step runs eagerly, then each pre-step state (arena permutation, speed flag) is captured once and
// replayed.
int advance(fs2d_batch* b) {
    if (b->prm.launch_mode == FS2D_LAUNCH_EAGER || b->steps_done == 0) {
        const int rc = step(b);
        if (rc == FS2D_OK) ++b->steps_done;
        return rc;
    }
    for (auto* g : b->graphs) {
        if (std::memcmp(g->pre, b->roles.a, sizeof g->pre) != 0 || g->pre_speed != b->speed_valid) continue;
        FS2D_BHIP(b, hipGraphLaunch(g->exec, b->stream));
        std::memcpy(b->roles.a, g->post, sizeof g->post);
        b->speed_valid = true;
        ++b->steps_done;
        return FS2D_OK;
    }
    if (b->graphs.size() >= kMaxBatchGraphs) drop_graphs(b);
    auto* g = new BatchGraph();
    std::memcpy(g->pre, b->roles.a, sizeof g->pre);
    g->pre_speed = b->speed_valid;
    hipError_t e = hipStreamBeginCapture(b->stream, hipStreamCaptureModeThreadLocal);
    if (e != hipSuccess) {
        delete g;
        return bfail(b, FS2D_ERR_HIP, std::string("hipStreamBeginCapture: ") + hipGetErrorString(e));
    }
    const int rc = step(b);
    e = hipStreamEndCapture(b->stream, &g->graph);
    if (rc == FS2D_OK && e == hipSuccess) e = hipGraphInstantiate(&g->exec, g->graph, nullptr, nullptr, 0);
    if (rc != FS2D_OK || e != hipSuccess) {
        std::memcpy(b->roles.a, g->pre, sizeof g->pre);  // nothing the capture recorded has run
        b->speed_valid = g->pre_speed;
        if (g->exec) (void)hipGraphExecDestroy(g->exec);
        if (g->graph) (void)hipGraphDestroy(g->graph);
        delete g;
        return rc != FS2D_OK ? rc : bfail(b, FS2D_ERR_HIP, std::string("batch graph capture: ") + hipGetErrorString(e));
    }
    std::memcpy(g->post, b->roles.a, sizeof g->post);
    b->graphs.push_back(g);
    FS2D_BHIP(b, hipGraphLaunch(g->exec, b->stream));
    ++b->steps_done;
    return FS2D_OK;
}

// Exceptions thrown on the host (allocation in plan building, maps and
// vectors) never cross the C ABI: they become an error code and message.
template <class F>
int guarded(fs2d_batch* h, const char* what, F&& body) {
    try {
        return body();
    } catch (const std::bad_alloc&) {
        return bfail(h, FS2D_ERR_HIP, std::string(what) + ": out of host memory");
    } catch (const std::exception& e) {
        return bfail(h, FS2D_ERR_STATE, std::string(what) + ": " + e.what());
    } catch (...) {
        return bfail(h, FS2D_ERR_STATE, std::string(what) + ": unexpected exception");
    }
}

}  // namespace

extern "C" {

int fs2d_hip_batch_destroy(fs2d_batch* b) {
    if (!b) return FS2D_OK;
    if (b->stream) (void)hipStreamSynchronize(b->stream);
    drop_graphs(b);
    if (b->jacobi.diffuse) (void)hipFree(b->jacobi.diffuse);
    if (b->jacobi.pressure) (void)hipFree(b->jacobi.pressure);
    if (b->jacobi.diffuse_strips) (void)hipFree(b->jacobi.diffuse_strips);
    if (b->jacobi.pressure_strips) (void)hipFree(b->jacobi.pressure_strips);
    for (float* p : b->roles.a)
        if (p) (void)hipFree(p);
    if (b->sims) (void)hipFree(b->sims);
    if (b->cell_work) (void)hipFree(b->cell_work);
    if (b->max_bits) (void)hipFree(b->max_bits);
    if (b->slots) (void)hipFree(b->slots);
    if (b->scatter_sims) (void)hipFree(b->scatter_sims);
    if (b->scatter_windows) (void)hipFree(b->scatter_windows);
    if (b->scatter_scratch) (void)hipFree(b->scatter_scratch);
    if (b->scatter_flag) (void)hipFree(b->scatter_flag);
    stage_free(b->stage);
    if (b->stream) (void)hipStreamDestroy(b->stream);
    delete b;
    return FS2D_OK;
}

static int fs2d_hip_batch_create_impl(int count, const fs2d_batch_sim* sims, const fs2d_params* params, fs2d_batch** out) {
    if (!out) return bfail(nullptr, FS2D_ERR_ARGUMENT, "fs2d_hip_batch_create: out is NULL");
    *out = nullptr;
    if (count < 1 || count > (1 << 20) || !sims)
        return bfail(nullptr, FS2D_ERR_ARGUMENT, "fs2d_hip_batch_create: count must be in [1, 2^20] with sims given");
    fs2d_params prm;
    fs2d_default_params(&prm);
    prm.sweep_order = FS2D_ORDER_JACOBI;
    if (params) prm = *params;
    if (prm.sweep_order != FS2D_ORDER_JACOBI)
        return bfail(nullptr, FS2D_ERR_ARGUMENT,
                     "fs2d_hip_batch_create: batches run the Jacobi order only (sweep_order must be FS2D_ORDER_JACOBI)");
    if (prm.launch_mode != FS2D_LAUNCH_GRAPH && prm.launch_mode != FS2D_LAUNCH_EAGER)
        return bfail(nullptr, FS2D_ERR_ARGUMENT, "fs2d_hip_batch_create: launch_mode must be 0 (graph) or 1 (eager)");
    for (int s = 0; s < count; ++s) {
        const fs2d_batch_sim& q = sims[s];
        if (q.rows < 3 || q.rows > 8194)
            return bfail(nullptr, FS2D_ERR_ARGUMENT, "fs2d_hip_batch_create: rows must be in [3, 8194]");
        if (q.iterations < 2 || q.iterations > 1000000)
            return bfail(nullptr, FS2D_ERR_ARGUMENT, "fs2d_hip_batch_create: iterations must be in [2, 1e6]");
    }
    if (prm.jacobi_block != 0) {
        const int m = prm.jacobi_block;
        bool ok = m == 1 || m == 2 || m == 4 || m == 8;
        for (int s = 0; s < count && ok; ++s) ok = sims[s].iterations % m == 0 && sims[s].iterations / m >= 2;
        if (!ok)
            return bfail(nullptr, FS2D_ERR_ARGUMENT,
                         "fs2d_hip_batch_create: jacobi_block must be 1, 2, 4 or 8 and divide every simulation's "
                         "iterations at least twice");
    }
    fs2d_batch* b = new fs2d_batch();
    b->count = count;
    b->prm = prm;
    b->host_sims.resize(count);
    size_t off = 0;
    std::vector<int2> cw, sw;  // single-pass stage blocks; the scatter's window-path waves
    std::vector<ScatterSim> ss(count);
    long long scatter_cells = 0, scatter_targets = 0;
    for (int s = 0; s < count; ++s) {
        BatchSim& S = b->host_sims[s];
        const fs2d_batch_sim& q = sims[s];
        S.R = q.rows;
        S.P = (q.rows + 63) / 64 * 64;
        S.off = off;
        off += static_cast<size_t>(S.R) * S.P;  // a multiple of 64 floats
        S.dt = q.dt;
        // scalars exactly as the one-grid handle computes them
        S.dt0 = std::sqrt(cells_of(S.R)) * q.dt;
        S.h = 1.0f / std::sqrt(cells_of(S.R));
        S.neg_half_h = -0.5f * S.h;
        S.a_rho = q.dt * cells_of(S.R) * q.diffusion_rate;
        S.a_vel = q.dt * cells_of(S.R) * q.viscosity;
        SweepArgs dr = sweep_args(nullptr, nullptr, S.R, S.P, SWEEP_DIFFUSE, S.a_rho, 1.f + 4.f * S.a_rho, BND_CONT, 2, 0);
        SweepArgs dv = sweep_args(nullptr, nullptr, S.R, S.P, SWEEP_DIFFUSE, S.a_vel, 1.f + 4.f * S.a_vel, BND_CONT, 2, 0);
        known_quotient(dr);
        known_quotient(dv);
        S.dv_rho = jac::divisor_of(dr);
        S.dv_vel = jac::divisor_of(dv);
        S.checked_rho = dr.div_checked;
        S.checked_vel = dv.div_checked;
        const int most = prm.jacobi_block ? prm.jacobi_block : jac::kTileMaxSweeps;
        S.launches = std::max(2, (q.iterations + most - 1) / most);
        S.sweeps = q.iterations / S.launches;
        S.longer = q.iterations % S.launches;
        const int n = S.R - 2;
        const int gx = (n + CBX - 1) / CBX, gy = (n + CBY - 1) / CBY;
        for (int by = 0; by < gy; ++by)
            for (int bx = 0; bx < gx; ++bx) cw.push_back(make_int2(s, (by << 16) | bx));
        ss[s] = ScatterSim{S.off, S.R, S.P, S.dt0, static_cast<unsigned>(scatter_cells),
                           static_cast<unsigned>(scatter_targets)};
        scatter_cells += static_cast<long long>(n) * n;
        scatter_targets += static_cast<long long>(S.R - 1) * (S.R - 1);
        for (int band = 0; band < (n + kBatchBand - 1) / kBatchBand; ++band)
            for (int strip = 0; strip < (n + kBatchStrip - 1) / kBatchStrip; ++strip)
                sw.push_back(make_int2(s, (band << 16) | strip));
        b->interior += static_cast<long long>(n) * n;
        b->order.push_back(s);
    }
    std::stable_sort(b->order.begin(), b->order.end(),
                     [&](int x, int y) { return b->host_sims[x].launches > b->host_sims[y].launches; });
    b->arena_floats = off;
    b->cell_blocks = static_cast<int>(cw.size());
    auto bail = [&](hipError_t e, const char* what) {
        std::string msg = std::string("fs2d_hip_batch_create: ") + what + ": " + hipGetErrorString(e);
        fs2d_hip_batch_destroy(b);
        return bfail(nullptr, FS2D_ERR_HIP, msg);
    };
    hipError_t e;
    if ((e = hipStreamCreateWithFlags(&b->stream, hipStreamNonBlocking)) != hipSuccess)
        return bail(e, "hipStreamCreate");
    {
        int dev = 0, cus = 0;
        if (hipGetDevice(&dev) == hipSuccess &&
            hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess && cus > 0)
            b->cus = cus;
    }
    const size_t bytes = sizeof(float) * off;
    const size_t fill_blocks = std::max<size_t>(1, std::min<size_t>((off + 255) / 256, 4096));
    for (int a = 0; a < A_COUNT; ++a) {
        if ((e = hipMalloc(&b->roles.a[a], bytes)) != hipSuccess) return bail(e, "hipMalloc(arena)");
        hipLaunchKernelGGL(kb_fill, dim3((unsigned)fill_blocks), dim3(256), 0, b->stream,
                           reinterpret_cast<uint32_t*>(b->roles.a[a]), off);
    }
    if ((e = hipMalloc(&b->sims, sizeof(BatchSim) * count)) != hipSuccess) return bail(e, "hipMalloc(sims)");
    if ((e = hipMalloc(&b->cell_work, sizeof(int2) * cw.size())) != hipSuccess) return bail(e, "hipMalloc(work)");
    if ((e = hipMalloc(&b->max_bits, sizeof(unsigned) * count)) != hipSuccess) return bail(e, "hipMalloc(speed)");
    const size_t slot_words = static_cast<size_t>(count) * kSimSlots * kSimSlotStride;
    if ((e = hipMalloc(&b->slots, sizeof(unsigned) * slot_words)) != hipSuccess) return bail(e, "hipMalloc(slots)");
    hipLaunchKernelGGL(kb_fill, dim3((unsigned)std::min<size_t>((slot_words + 255) / 256, 4096)), dim3(256), 0,
                       b->stream, b->slots, slot_words);
    if ((e = build_jacobi_work(b)) != hipSuccess) return bail(e, "Jacobi work lists");
    // the density scatter: descriptors, window work list, sorted-path buffers
    if (scatter_cells >= (1ll << 31) || scatter_targets >= (1ll << 32) - 1)
        return bail(hipErrorInvalidValue, "too many cells for the batched density scatter");
    if ((e = hipMalloc(&b->scatter_sims, sizeof(ScatterSim) * count)) != hipSuccess)
        return bail(e, "hipMalloc(scatter descriptors)");
    if ((e = hipMalloc(&b->scatter_windows, sizeof(int2) * sw.size())) != hipSuccess)
        return bail(e, "hipMalloc(scatter work)");
    if ((e = hipMalloc(&b->scatter_scratch, batch_scatter_bytes(scatter_cells, scatter_targets))) != hipSuccess)
        return bail(e, "hipMalloc(scatter buffers)");
    if ((e = hipMalloc(&b->scatter_flag, 256)) != hipSuccess) return bail(e, "hipMalloc(scatter gate)");
    if ((e = hipMemcpyAsync(b->scatter_sims, ss.data(), sizeof(ScatterSim) * count, hipMemcpyHostToDevice,
                            b->stream)) != hipSuccess)
        return bail(e, "hipMemcpy(scatter descriptors)");
    if ((e = hipMemcpyAsync(b->scatter_windows, sw.data(), sizeof(int2) * sw.size(), hipMemcpyHostToDevice,
                            b->stream)) != hipSuccess)
        return bail(e, "hipMemcpy(scatter work)");
    b->scatter = BatchScatter{b->scatter_sims, count, b->scatter_windows, static_cast<int>(sw.size()), scatter_cells,
                              scatter_targets, b->scatter_scratch, b->scatter_flag};
    if ((e = hipMemcpyAsync(b->cell_work, cw.data(), sizeof(int2) * cw.size(), hipMemcpyHostToDevice, b->stream)) !=
        hipSuccess)
        return bail(e, "hipMemcpy(work)");
    if ((e = hipMemcpyAsync(b->sims, b->host_sims.data(), sizeof(BatchSim) * count, hipMemcpyHostToDevice,
                            b->stream)) != hipSuccess)
        return bail(e, "hipMemcpy(sims)");
    if ((e = hipStreamSynchronize(b->stream)) != hipSuccess) return bail(e, "hipStreamSynchronize");
    *out = b;
    return FS2D_OK;
}

int fs2d_hip_batch_create(int count, const fs2d_batch_sim* sims, const fs2d_params* params, fs2d_batch** out) {
    return guarded(nullptr, "fs2d_hip_batch_create", [&] { return fs2d_hip_batch_create_impl(count, sims, params, out); });
}

static int fs2d_hip_batch_upload_impl(fs2d_batch* b, int sim, const float* rho, const float* u, const float* v) {
    if (!b || sim < 0 || sim >= (b ? b->count : 0) || !rho || !u || !v)
        return bfail(b, FS2D_ERR_ARGUMENT, "fs2d_hip_batch_upload: bad argument");
    const BatchSim& S = b->host_sims[sim];
    RowCopies c;
    c.add(rho, b->roles.a[A_RHO] + S.off);
    c.add(u, b->roles.a[A_U] + S.off);
    c.add(v, b->roles.a[A_V] + S.off);
    b->speed_valid = false;
    FS2D_BHIP(b, stage_in(b->stage, b->stream, c, S.R, S.P));
    FS2D_BHIP(b, hipStreamSynchronize(b->stream));
    return FS2D_OK;
}

int fs2d_hip_batch_upload(fs2d_batch* b, int sim, const float* rho, const float* u, const float* v) {
    return guarded(b, "fs2d_hip_batch_upload", [&] { return fs2d_hip_batch_upload_impl(b, sim, rho, u, v); });
}

static int fs2d_hip_batch_set_sources_impl(fs2d_batch* b, int sim, const float* rs, const float* us, const float* vs) {
    if (!b || sim < 0 || sim >= b->count) return bfail(b, FS2D_ERR_ARGUMENT, "fs2d_hip_batch_set_sources: bad argument");
    const float* src[3] = {rs, us, vs};
    const int dst[3] = {A_RS, A_US, A_VS};
    const BatchSim& S = b->host_sims[sim];
    const size_t n = static_cast<size_t>(S.R) * S.P;
    RowCopies c;
    for (int i = 0; i < 3; ++i) {
        if (src[i]) {
            c.add(src[i], b->roles.a[dst[i]] + S.off);
        } else {
            hipLaunchKernelGGL(kb_fill, dim3((unsigned)std::max<size_t>(1, std::min<size_t>((n + 255) / 256, 4096))),
                               dim3(256), 0, b->stream, reinterpret_cast<uint32_t*>(b->roles.a[dst[i]] + S.off), n);
            FS2D_BHIP(b, hipGetLastError());
        }
    }
    FS2D_BHIP(b, stage_in(b->stage, b->stream, c, S.R, S.P));
    FS2D_BHIP(b, hipStreamSynchronize(b->stream));
    return FS2D_OK;
}

int fs2d_hip_batch_set_sources(fs2d_batch* b, int sim, const float* rs, const float* us, const float* vs) {
    return guarded(b, "fs2d_hip_batch_set_sources", [&] { return fs2d_hip_batch_set_sources_impl(b, sim, rs, us, vs); });
}

static int fs2d_hip_batch_step_n_impl(fs2d_batch* b, int n) {
    if (!b || n < 0) return bfail(b, FS2D_ERR_ARGUMENT, "fs2d_hip_batch_step_n: bad argument");
    for (int i = 0; i < n; ++i) {
        const int rc = advance(b);
        if (rc) return rc;
    }
    return FS2D_OK;
}

int fs2d_hip_batch_step_n(fs2d_batch* b, int n) {
    return guarded(b, "fs2d_hip_batch_step_n", [&] { return fs2d_hip_batch_step_n_impl(b, n); });
}

static int fs2d_hip_batch_download_impl(fs2d_batch* b, int sim, float* rho, float* u, float* v) {
    if (!b || sim < 0 || sim >= b->count) return bfail(b, FS2D_ERR_ARGUMENT, "fs2d_hip_batch_download: bad argument");
    const BatchSim& S = b->host_sims[sim];
    RowCopies c;
    if (rho) c.add(b->roles.a[A_RHO] + S.off, rho);
    if (u) c.add(b->roles.a[A_U] + S.off, u);
    if (v) c.add(b->roles.a[A_V] + S.off, v);
    FS2D_BHIP(b, stage_out(b->stage, b->stream, c, S.R, S.P));
    return FS2D_OK;
}

int fs2d_hip_batch_download(fs2d_batch* b, int sim, float* rho, float* u, float* v) {
    return guarded(b, "fs2d_hip_batch_download", [&] { return fs2d_hip_batch_download_impl(b, sim, rho, u, v); });
}

static int fs2d_hip_batch_sync_impl(fs2d_batch* b) {
    if (!b) return bfail(b, FS2D_ERR_ARGUMENT, "fs2d_hip_batch_sync: NULL batch");
    FS2D_BHIP(b, hipStreamSynchronize(b->stream));
    return FS2D_OK;
}

int fs2d_hip_batch_sync(fs2d_batch* b) {
    return guarded(b, "fs2d_hip_batch_sync", [&] { return fs2d_hip_batch_sync_impl(b); });
}

static int fs2d_hip_batch_info_impl(fs2d_batch* b, int* depth, int* tile_rows, int* launches, int* graphs,
                        long long* interior_cells) {
    if (!b) return bfail(b, FS2D_ERR_ARGUMENT, "fs2d_hip_batch_info: NULL batch");
    if (depth) *depth = b->prm.jacobi_block ? b->prm.jacobi_block : 1;
    if (tile_rows) *tile_rows = b->jacobi.rows - 2 * jac::kTileMaxSweeps;
    if (launches) {
        // max speed (first step only) aside, the passes of a step: add, diffuse launches, the scatter's
        // kernels, 2 x (divergence, pressure launches, gradient, fold), gather; adds and divergences made by first launches
        const int d = static_cast<int>(b->jacobi.diffuse_count.size());
        const int p = static_cast<int>(b->jacobi.pressure_count.size());
        *launches = b->steps_done > 0 ? 1 + d + batch_scatter_launches(b->scatter.targets) + 2 * (3 + p) + 1 : 0;
    }
    if (graphs) *graphs = static_cast<int>(b->graphs.size());
    if (interior_cells) *interior_cells = b->interior;
    return FS2D_OK;
}

// As fs2d_hip_step_launches.
static int fs2d_hip_batch_step_launches_impl(fs2d_batch* b, int* launches, int* fewest, int* most) {
    if (!b) return bfail(b, FS2D_ERR_ARGUMENT, "fs2d_hip_batch_step_launches: NULL batch");
    if (launches) {
        float* kept[A_COUNT];
        std::memcpy(kept, b->roles.a, sizeof kept);
        const bool speed = b->speed_valid;
        FS2D_BHIP(b, hipStreamBeginCapture(b->stream, hipStreamCaptureModeThreadLocal));
        const int rc = step(b);
        hipGraph_t graph = nullptr;
        size_t n = 0;
        hipError_t e = hipStreamEndCapture(b->stream, &graph);
        if (e == hipSuccess) e = hipGraphGetNodes(graph, nullptr, &n);
        if (graph) (void)hipGraphDestroy(graph);
        std::memcpy(b->roles.a, kept, sizeof kept);  // nothing of it has run
        b->speed_valid = speed;
        if (rc) return rc;
        FS2D_BHIP(b, e);
        *launches = static_cast<int>(n);
    }
    int lo = b->host_sims[0].sweeps, hi = 0;
    for (const BatchSim& S : b->host_sims) {
        lo = std::min(lo, S.sweeps);
        hi = std::max(hi, S.sweeps + (S.longer > 0));
    }
    if (fewest) *fewest = lo;
    if (most) *most = hi;
    return FS2D_OK;
}

int fs2d_hip_batch_step_launches(fs2d_batch* b, int* launches, int* fewest_sweeps, int* most_sweeps) {
    return guarded(b, "fs2d_hip_batch_step_launches", [&] { return fs2d_hip_batch_step_launches_impl(b, launches, fewest_sweeps, most_sweeps); });
}

int fs2d_hip_batch_set_occupancy(fs2d_batch* b, int jacobi_blocks_per_cu, int stage_blocks_per_cu) {
    if (!b || jacobi_blocks_per_cu < 0 || jacobi_blocks_per_cu > 64 || stage_blocks_per_cu < 0 ||
        stage_blocks_per_cu > 64)
        return bfail(b, FS2D_ERR_ARGUMENT, "fs2d_hip_batch_set_occupancy: blocks per CU must be in [0, 64]");
    if (b->steps_done > 0)
        return bfail(b, FS2D_ERR_STATE, "fs2d_hip_batch_set_occupancy: only before the first step");
    b->jac_per_cu = jacobi_blocks_per_cu;
    b->cell_per_cu = stage_blocks_per_cu;
    return FS2D_OK;
}

int fs2d_hip_batch_occupancy(fs2d_batch* b, int* jacobi_blocks_per_cu, int* stage_blocks_per_cu,
                             int* compute_units) {
    if (!b) return bfail(b, FS2D_ERR_ARGUMENT, "fs2d_hip_batch_occupancy: NULL batch");
    if (jacobi_blocks_per_cu) *jacobi_blocks_per_cu = b->jac_per_cu;
    if (stage_blocks_per_cu) *stage_blocks_per_cu = b->cell_per_cu;
    if (compute_units) *compute_units = b->cus;
    return FS2D_OK;
}

int fs2d_hip_batch_info(fs2d_batch* b, int* depth, int* tile_rows, int* launches, int* graphs,
                        long long* interior_cells) {
    return guarded(b, "fs2d_hip_batch_info", [&] { return fs2d_hip_batch_info_impl(b, depth, tile_rows, launches, graphs, interior_cells); });
}

const char* fs2d_hip_batch_last_error(const fs2d_batch* b) {
    return b ? b->err.c_str() : g_batch_create_error.c_str();
}

}  // extern "C"
