// fs2d_cnn_kernels.hpp -- device kernels of the pressure-guess network.
//
// Activations are NHWC bfloat16 with a channel count that is a multiple of
// 16; pixel p = (n * H + y) * W + x.  A 3x3 convolution (zero padding,
// stride 1) is an implicit GEMM D[co][p] = sum_{tap, ci} Wt[tap][co][ci] *
// X[p + tap][ci] on v_mfma_f32_16x16x16bf16_1k: lane l supplies
// A[m = l % 16][k = 4 (l / 16) + i] and B[k = 4 (l / 16) + i][n = l % 16] and
// holds D[m = 4 (l / 16) + i][n = l % 16], i = 0..3 (the network built from
// these kernels is checked on the device against a PyTorch reference).  With
// the output channels as rows, a lane ends with 4 consecutive channels of one
// pixel: one 8-byte store, and a wave's stores cover whole pixels.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace fs2d {
namespace cnn {

typedef uint16_t bf16;
typedef short short4_t __attribute__((ext_vector_type(4)));
typedef float float4_t __attribute__((ext_vector_type(4)));

__host__ __device__ inline float bf2f(bf16 b) {
    const uint32_t u = static_cast<uint32_t>(b) << 16;
    float f;
    __builtin_memcpy(&f, &u, 4);
    return f;
}

// Round to nearest even; NaN stays a quiet NaN.
__host__ __device__ inline bf16 f2bf(float f) {
    uint32_t u;
    __builtin_memcpy(&u, &f, 4);
    if ((u & 0x7fffffffu) > 0x7f800000u) return static_cast<bf16>((u >> 16) | 0x40u);
    u += 0x7fffu + ((u >> 16) & 1u);
    return static_cast<bf16>(u >> 16);
}

constexpr int CONV_WAVES = 4;  // waves per block

typedef short short8_t __attribute__((ext_vector_type(8)));

// What a convolution does with a pixel's 4 consecutive outputs co .. co + 3.
// y holds channels [0, Ca) of every pixel, y2 the channels [Ca, Cout) (the two
// parts of a concatenation's gradient; Ca = Cout and y2 unused otherwise).
// relu applies max(., 0); mask (Cout channels, may be null) zeroes the
// outputs whose value there is not > 0 (the derivative of the ReLU that
// made it).  OUT_F32: only channel 0, in fp32, one float a pixel (the
// network's one real output channel).
struct ConvOut {
    void* y;
    bf16* y2;
    const bf16* mask;
    const float* bias;
    int Cout, Ca, relu;
};

template <bool OUT_F32>
__device__ __forceinline__ void conv_store(const ConvOut& o, long p, int co, float4_t acc) {
    if (OUT_F32) {
        if (co == 0) static_cast<float*>(o.y)[p] = o.bias ? acc[0] + o.bias[0] : acc[0];
        return;
    }
    float4_t b = {0.f, 0.f, 0.f, 0.f};
    if (o.bias) b = *reinterpret_cast<const float4_t*>(o.bias + co);
    short4_t r;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        float v = acc[i] + b[i];
        if (o.relu) v = fmaxf(v, 0.f);
        r[i] = static_cast<short>(f2bf(v));
    }
    if (o.mask) {
        const short4_t m = *reinterpret_cast<const short4_t*>(o.mask + p * o.Cout + co);
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (!(bf2f(static_cast<bf16>(m[i])) > 0.f)) r[i] = 0;
    }
    bf16* q = co < o.Ca ? static_cast<bf16*>(o.y) + p * o.Ca + co : o.y2 + p * (o.Cout - o.Ca) + co - o.Ca;
    *reinterpret_cast<short4_t*>(q) = r;
}

// 3x3 convolution with both operands from global memory, NT output-channel
// tiles of 16 per wave, 16 pixels per wave: for images that do not tile into
// 8 x 16 pixels (the coarse levels of small or odd fields).
template <int NT, bool OUT_F32>
__global__ __launch_bounds__(64 * CONV_WAVES) void k_conv3x3(const bf16* __restrict__ x, int N, int H, int W, int Cin,
                                                            const bf16* __restrict__ w, ConvOut o) {
    const int wave = threadIdx.x >> 6, l = threadIdx.x & 63;
    const int Cout = o.Cout;
    const long npix = static_cast<long>(N) * H * W;
    const long p0 = (static_cast<long>(blockIdx.x) * CONV_WAVES + wave) * 16;
    if (p0 >= npix) return;  // whole wave; npix is a multiple of 16
    const int co0 = blockIdx.y * 16 * NT;
    const long pa = p0 + (l & 15);
    const int xa = static_cast<int>(pa % W);
    const long t0 = pa / W;
    const int ya = static_cast<int>(t0 % H);
    const long na = t0 / H;
    const int kq = (l >> 4) * 4;
    float4_t acc[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) acc[t] = float4_t{0.f, 0.f, 0.f, 0.f};
    for (int tap = 0; tap < 9; ++tap) {
        const int yy = ya + tap / 3 - 1, xx = xa + tap % 3 - 1;
        const bool in = (unsigned)yy < (unsigned)H && (unsigned)xx < (unsigned)W;
        // clamped address: always inside the tensor; out-of-image taps read zero
        const int yc = min(max(yy, 0), H - 1), xc = min(max(xx, 0), W - 1);
        const bf16* xp = x + ((na * H + yc) * W + xc) * Cin + kq;
        const bf16* wp = w + (static_cast<long>(tap) * Cout + co0 + (l & 15)) * Cin + kq;
        for (int c0 = 0; c0 < Cin; c0 += 16) {
            short4_t a = *reinterpret_cast<const short4_t*>(xp + c0);
            if (!in) a = short4_t{0, 0, 0, 0};
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                const short4_t b = *reinterpret_cast<const short4_t*>(wp + static_cast<long>(t) * 16 * Cin + c0);
                acc[t] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(b, a, acc[t], 0, 0, 0);
            }
        }
    }
#pragma unroll
    for (int t = 0; t < NT; ++t) conv_store<OUT_F32>(o, pa, co0 + 16 * t + kq, acc[t]);
}

// The same convolution with the operands staged in LDS.  A block computes a
// 4G-row x 16-column pixel tile (W a multiple of 16) for 16 NT output channels;
// wave w takes rows G w .. G w + G - 1, so each weight fragment feeds G MFMAs
// and each pixel fragment NT.  Per 16-channel input chunk the block stages the
// tile's (4G + 2) x 18 input halo (zero outside the image) and the chunk's
// 9 x 16 NT x 16 weights.  Two buffers: a chunk's loads are in flight, in
// registers, while the one before is multiplied, and one barrier separates
// two chunks.  LDS holds 4 planes of 4 channels each: the 16 lanes that read
// 4 channels of 16 neighbouring pixels touch 128 contiguous bytes, and planes
// lie 128 bytes apart modulo the 256 of all banks.
template <int NT, int G, bool OUT_F32>
__global__ __launch_bounds__(256) void k_conv3x3_lds(const bf16* __restrict__ x, int N, int H, int W, int Cin,
                                                    const bf16* __restrict__ w, ConvOut o) {
    constexpr int TR = 4 * G, TC = 16, HR = TR + 2, HC = TC + 2;
    constexpr int CO = 16 * NT;
    constexpr int XP = HR * HC, WP = 9 * CO;  // pixels and weight rows per plane
    constexpr int XS = (XP + 15) / 32 * 32 + 16, WS = (WP + 15) / 32 * 32 + 16;  // plane strides
    constexpr int XI = (2 * XP + 255) / 256, WI = (2 * WP + 255) / 256;          // 16-byte items per thread
    __shared__ short4_t xs[2][4 * XS];
    __shared__ short4_t ws[2][4 * WS];
    const int tid = threadIdx.x, wave = tid >> 6, l = tid & 63;
    const int tiles_x = W / TC, tiles_y = (H + TR - 1) / TR;
    int b = blockIdx.x;
    const int tx = b % tiles_x;
    b /= tiles_x;
    const int ty = b % tiles_y;
    const long n = b / tiles_y;
    const int x0 = tx * TC, y0 = ty * TR;
    const int Cout = o.Cout, co0 = blockIdx.y * CO;
    const int kq4 = l >> 4;  // which plane this lane reads
    short8_t xr[XI], wr[WI];
    auto load = [&](int c0) {
#pragma unroll
        for (int k = 0; k < XI; ++k) {
            const int q = tid + 256 * k, half = q & 1, pix = q >> 1;
            const int yy = y0 + pix / HC - 1, xx = x0 + pix % HC - 1;
            xr[k] = short8_t{0, 0, 0, 0, 0, 0, 0, 0};
            if (pix < XP && (unsigned)yy < (unsigned)H && (unsigned)xx < (unsigned)W)
                xr[k] = *reinterpret_cast<const short8_t*>(x + ((n * H + yy) * W + xx) * Cin + c0 + 8 * half);
        }
#pragma unroll
        for (int k = 0; k < WI; ++k) {
            const int q = tid + 256 * k, half = q & 1, tc = q >> 1;
            if (tc < WP)
                wr[k] = *reinterpret_cast<const short8_t*>(
                    w + (static_cast<long>(tc / CO) * Cout + co0 + tc % CO) * Cin + c0 + 8 * half);
        }
    };
    auto store = [&](int buf) {
#pragma unroll
        for (int k = 0; k < XI; ++k) {
            const int q = tid + 256 * k, half = q & 1, pix = q >> 1;
            if (pix < XP) {
                xs[buf][(2 * half) * XS + pix] = __builtin_shufflevector(xr[k], xr[k], 0, 1, 2, 3);
                xs[buf][(2 * half + 1) * XS + pix] = __builtin_shufflevector(xr[k], xr[k], 4, 5, 6, 7);
            }
        }
#pragma unroll
        for (int k = 0; k < WI; ++k) {
            const int q = tid + 256 * k, half = q & 1, tc = q >> 1;
            if (tc < WP) {
                ws[buf][(2 * half) * WS + tc] = __builtin_shufflevector(wr[k], wr[k], 0, 1, 2, 3);
                ws[buf][(2 * half + 1) * WS + tc] = __builtin_shufflevector(wr[k], wr[k], 4, 5, 6, 7);
            }
        }
    };
    float4_t acc[G][NT];
#pragma unroll
    for (int g = 0; g < G; ++g)
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[g][t] = float4_t{0.f, 0.f, 0.f, 0.f};
    load(0);
    store(0);
    __syncthreads();
    for (int c0 = 0, buf = 0; c0 < Cin; c0 += 16, buf ^= 1) {
        const bool more = c0 + 16 < Cin;
        if (more) load(c0 + 16);
        const short4_t* xb = xs[buf] + kq4 * XS + (l & 15);
        const short4_t* wb = ws[buf] + kq4 * WS + (l & 15);
#pragma unroll
        for (int tap = 0; tap < 9; ++tap) {
            const int dy = tap / 3, dx = tap % 3;  // offsets into the halo (0..2)
            short4_t a[G];
#pragma unroll
            for (int g = 0; g < G; ++g) a[g] = xb[(G * wave + g + dy) * HC + dx];
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                const short4_t bb = wb[tap * CO + 16 * t];
#pragma unroll
                for (int g = 0; g < G; ++g)
                    acc[g][t] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(bb, a[g], acc[g][t], 0, 0, 0);
            }
        }
        if (more) {
            store(buf ^ 1);
            __syncthreads();
        }
    }
#pragma unroll
    for (int g = 0; g < G; ++g) {
        const int yy = y0 + G * wave + g;
        if (yy >= H) continue;
        const long p = (n * H + yy) * W + x0 + (l & 15);
#pragma unroll
        for (int t = 0; t < NT; ++t) conv_store<OUT_F32>(o, p, co0 + 16 * t + 4 * kq4, acc[g][t]);
    }
}

// Weight gradient gw[tap][co][ci] = sum_p dz[p][co] * x[p + tap][ci] and bias
// gradient gb[co] = sum_p dz[p][co], as partial sums over the pixel tiles that
// a block walks: a GEMM whose inner dimension is the pixels.
//
// A block takes 16 NA output channels x 16 NB input channels of all 9 taps
// (36 NA NB accumulators a lane) and the 16 x 32 pixel tiles blockIdx.x,
// blockIdx.x + splits, ...; wave w takes 4 rows of 16 columns of each tile.  The
// tile of dz and the halo of x lie in LDS as 16-channel rows, one a pixel, and
// ds_read_tr16_b64 reads fragments across the pixels, so a tap is an offset of
// whole rows.  An MFMA takes 32 pixels: 16 columns of two neighbouring rows
// (the order of the inner dimension is free as long as both operands share
// it), and the 4 x 3 pixel fragments that a lane holds serve all 9 taps of both
// rows.  The next tile's loads are in flight, in registers, meanwhile.  Pixels
// outside the image are zero in both operands.
//
// The 8 waves' accumulators are added in LDS, a tap at a time, and each block
// writes its sums to part[split] (weights [9][Cout][Cin], then Cout biases); k_reduce_adam
// adds the splits.  No atomics: the gradients are the same bits on every run.
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));

constexpr int WG_R = 16, WG_C = 32, WG_THREADS = 512;

template <int NA, int NB>
__global__ __launch_bounds__(WG_THREADS) void k_conv3x3_wgrad(const bf16* __restrict__ x, const bf16* __restrict__ dz,
                                                             int N, int H, int W, int Cin, int Cout,
                                                             float* __restrict__ part) {
    constexpr int HR = WG_R + 2, HC = WG_C + 2, XP = HR * HC, ZP = WG_R * WG_C;
    constexpr int XI = (2 * NB * XP + WG_THREADS - 1) / WG_THREADS, ZI = 2 * NA * ZP / WG_THREADS;
    constexpr int kTile = (NB * XP + NA * ZP) * 16, kSum = 8 * NA * NB * 256 * 2;  // in bf16
    __shared__ bf16 sm[kTile > kSum ? kTile : kSum] __attribute__((aligned(16)));
    bf16* const xs = sm;                     // [NB][XP][16]
    bf16* const zs = sm + NB * XP * 16;      // [NA][ZP][16]
    const int tid = threadIdx.x, wave = tid >> 6, l = tid & 63;
    const int nci = Cin / (16 * NB);
    const int ci0 = (blockIdx.y % nci) * 16 * NB, co0 = (blockIdx.y / nci) * 16 * NA;
    const int tiles_x = (W + WG_C - 1) / WG_C, tiles_y = (H + WG_R - 1) / WG_R;
    const int tiles = N * tiles_y * tiles_x;
    short8_t xr[XI], zr[ZI];
    auto load = [&](int tile) {
        const int tx = tile % tiles_x, r = tile / tiles_x;
        const int y0 = (r % tiles_y) * WG_R, x0 = tx * WG_C;
        const long n = r / tiles_y;
#pragma unroll
        for (int k = 0; k < XI; ++k) {
            const int q = tid + WG_THREADS * k, part8 = q % (2 * NB), pix = q / (2 * NB);
            const int yy = y0 + pix / HC - 1, xx = x0 + pix % HC - 1;
            xr[k] = short8_t{0, 0, 0, 0, 0, 0, 0, 0};
            if (pix < XP && (unsigned)yy < (unsigned)H && (unsigned)xx < (unsigned)W)
                xr[k] = *reinterpret_cast<const short8_t*>(x + ((n * H + yy) * W + xx) * Cin + ci0 + 8 * part8);
        }
#pragma unroll
        for (int k = 0; k < ZI; ++k) {
            const int q = tid + WG_THREADS * k, part8 = q % (2 * NA), pix = q / (2 * NA);
            const int yy = y0 + pix / WG_C, xx = x0 + pix % WG_C;
            zr[k] = short8_t{0, 0, 0, 0, 0, 0, 0, 0};
            if (yy < H && xx < W)
                zr[k] = *reinterpret_cast<const short8_t*>(dz + ((n * H + yy) * W + xx) * Cout + co0 + 8 * part8);
        }
    };
    auto store = [&]() {
#pragma unroll
        for (int k = 0; k < XI; ++k) {
            const int q = tid + WG_THREADS * k, part8 = q % (2 * NB), pix = q / (2 * NB);
            if (pix < XP) *reinterpret_cast<short8_t*>(xs + ((part8 >> 1) * XP + pix) * 16 + 8 * (part8 & 1)) = xr[k];
        }
#pragma unroll
        for (int k = 0; k < ZI; ++k) {
            const int q = tid + WG_THREADS * k, part8 = q % (2 * NA), pix = q / (2 * NA);
            *reinterpret_cast<short8_t*>(zs + ((part8 >> 1) * ZP + pix) * 16 + 8 * (part8 & 1)) = zr[k];
        }
    };
    // Lane l of 16-lane group g reads 4 channels of pixel 4 g + (l % 16) / 4 and
    // receives channel l % 16 of pixels 4 g .. 4 g + 3.
    const int lane_off = (4 * (l >> 4) + ((l & 15) >> 2)) * 16 + 4 * (l & 3);
    typedef __attribute__((address_space(3))) short4_t* lds_ptr;
    auto frag = [&](const bf16* base) { return __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)(base + lane_off)); };
    auto pair = [](short4_t lo, short4_t hi) {
        return __builtin_bit_cast(bf16x8_t, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
    };
    float4_t acc[9][NA][NB], accb[NA];
#pragma unroll
    for (int t = 0; t < 9; ++t)
#pragma unroll
        for (int a = 0; a < NA; ++a)
#pragma unroll
            for (int b = 0; b < NB; ++b) acc[t][a][b] = float4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int a = 0; a < NA; ++a) accb[a] = float4_t{0.f, 0.f, 0.f, 0.f};
    const short4_t one4 = {0x3f80, 0x3f80, 0x3f80, 0x3f80};
    const bf16x8_t ones = pair(one4, one4);
    const int c16 = 16 * (wave & 1), r4 = 4 * (wave >> 1);

    int tile = blockIdx.x;
    if (tile < tiles) load(tile);
    for (; tile < tiles; tile += gridDim.x) {
        __syncthreads();  // the previous tile's reads are done
        store();
        __syncthreads();
        if (tile + (int)gridDim.x < tiles) load(tile + gridDim.x);
#pragma unroll
        for (int r = 0; r < 4; r += 2) {
            bf16x8_t z[NA];
#pragma unroll
            for (int a = 0; a < NA; ++a)
                z[a] = pair(frag(zs + (a * ZP + (r4 + r) * WG_C + c16) * 16),
                            frag(zs + (a * ZP + (r4 + r + 1) * WG_C + c16) * 16));
#pragma unroll
            for (int b = 0; b < NB; ++b) {
                short4_t f[4][3];
#pragma unroll
                for (int h = 0; h < 4; ++h)
#pragma unroll
                    for (int dx = 0; dx < 3; ++dx)
                        f[h][dx] = frag(xs + (b * XP + (r4 + r + h) * HC + c16 + dx) * 16);
#pragma unroll
                for (int t = 0; t < 9; ++t) {
                    const bf16x8_t xx = pair(f[t / 3][t % 3], f[t / 3 + 1][t % 3]);
#pragma unroll
                    for (int a = 0; a < NA; ++a)
                        acc[t][a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(z[a], xx, acc[t][a][b], 0, 0, 0);
                }
            }
#pragma unroll
            for (int a = 0; a < NA; ++a) accb[a] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(z[a], ones, accb[a], 0, 0, 0);
        }
    }

    // D[m = 4 (l / 16) + i][n = l % 16]: output channel m, input channel n.
    float* const fs = reinterpret_cast<float*>(sm);  // [8 waves][NA * NB][256]
    float* const out = part + static_cast<long>(blockIdx.x) * (9L * Cin * Cout + Cout);
    for (int t = 0; t < 9; ++t) {
        __syncthreads();
#pragma unroll
        for (int tt = 0; tt < 9; ++tt)
            if (tt == t) {
#pragma unroll
                for (int a = 0; a < NA; ++a)
#pragma unroll
                    for (int b = 0; b < NB; ++b)
#pragma unroll
                        for (int i = 0; i < 4; ++i)
                            fs[((wave * NA + a) * NB + b) * 256 + (4 * (l >> 4) + i) * 16 + (l & 15)] = acc[tt][a][b][i];
            }
        __syncthreads();
        for (int q = tid; q < NA * NB * 256; q += WG_THREADS) {
            float sum = 0.f;
#pragma unroll
            for (int v = 0; v < 8; ++v) sum += fs[v * NA * NB * 256 + q];
            const int n = q & 15, m = (q >> 4) & 15, b = (q >> 8) % NB, a = (q >> 8) / NB;
            out[(static_cast<long>(t) * Cout + co0 + 16 * a + m) * Cin + ci0 + 16 * b + n] = sum;
        }
    }
    if (ci0 != 0) return;
    __syncthreads();
    if ((l & 15) == 0) {
#pragma unroll
        for (int a = 0; a < NA; ++a)
#pragma unroll
            for (int i = 0; i < 4; ++i) fs[wave * 16 * NA + 16 * a + 4 * (l >> 4) + i] = accb[a][i];
    }
    __syncthreads();
    if (tid < 16 * NA) {
        float sum = 0.f;
#pragma unroll
        for (int v = 0; v < 8; ++v) sum += fs[v * 16 * NA + tid];
        out[9L * Cin * Cout + co0 + tid] = sum;
    }
}

// wt[8 - tap][ci][co] = w[tap][co][ci]: the weights of the data gradient (a
// 3x3 convolution of dz with the flipped, transposed kernel).
__global__ __launch_bounds__(256) void k_flip_weights(const bf16* __restrict__ w, bf16* __restrict__ wt, int Cin,
                                                     int Cout) {
    const long n = 9L * Cin * Cout;
    for (long t = static_cast<long>(blockIdx.x) * 256 + threadIdx.x; t < n; t += static_cast<long>(gridDim.x) * 256) {
        const int ci = static_cast<int>(t % Cin);
        const long r = t / Cin;
        const int co = static_cast<int>(r % Cout);
        const int tap = static_cast<int>(r / Cout);
        wt[(static_cast<long>(8 - tap) * Cin + ci) * Cout + co] = w[t];
    }
}

// 2x2 average: y[n][i][j][c] from x[n][2i..2i+1][2j..2j+1][c].  A thread takes
// 8 channels (16-byte accesses), as do the kernels below: these passes are bound
// by memory, and by the address arithmetic when it is done per channel.
__global__ __launch_bounds__(256) void k_avgpool2(const bf16* __restrict__ x, bf16* __restrict__ y, int N, int H, int W,
                                                 int C) {
    const int h = H / 2, w = W / 2, G = C / 8;
    const long n = static_cast<long>(N) * h * w * G;
    for (long t = static_cast<long>(blockIdx.x) * 256 + threadIdx.x; t < n; t += static_cast<long>(gridDim.x) * 256) {
        const int g = static_cast<int>(t % G);
        long r = t / G;
        const int j = static_cast<int>(r % w);
        r /= w;
        const int i = static_cast<int>(r % h);
        const long b = r / h;
        const bf16* q = x + ((b * H + 2 * i) * W + 2 * j) * C + 8 * g;
        const short8_t a0 = *reinterpret_cast<const short8_t*>(q), a1 = *reinterpret_cast<const short8_t*>(q + C);
        const short8_t b0 = *reinterpret_cast<const short8_t*>(q + static_cast<long>(W) * C);
        const short8_t b1 = *reinterpret_cast<const short8_t*>(q + static_cast<long>(W) * C + C);
        short8_t out;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const float s = (bf2f(static_cast<bf16>(a0[e])) + bf2f(static_cast<bf16>(a1[e]))) +
                            (bf2f(static_cast<bf16>(b0[e])) + bf2f(static_cast<bf16>(b1[e])));
            out[e] = static_cast<short>(f2bf(0.25f * s));
        }
        *reinterpret_cast<short8_t*>(y + t * 8) = out;
    }
}

// r where mask > 0, else 0: the derivative of the ReLU whose output mask is.
__device__ __forceinline__ short8_t relu_masked(short8_t r, const bf16* __restrict__ mask) {
    const short8_t m = *reinterpret_cast<const short8_t*>(mask);
#pragma unroll
    for (int e = 0; e < 8; ++e)
        if (!(bf2f(static_cast<bf16>(m[e])) > 0.f)) r[e] = 0;
    return r;
}

// out[n][y][x][c] = dy[n][y/2][x/2][c] / 4 + skip[n][y][x][c]: the pool's
// backward, summed with the gradient the same activation gets through its
// skip connection, then through the activation's ReLU (its output is mask).
__global__ __launch_bounds__(256) void k_pool_bwd_add(const bf16* __restrict__ dy, const bf16* __restrict__ skip,
                                                     const bf16* __restrict__ mask, bf16* __restrict__ out, int N,
                                                     int H, int W, int C) {
    const int G = C / 8;
    const long n = static_cast<long>(N) * H * W * G;
    for (long t = static_cast<long>(blockIdx.x) * 256 + threadIdx.x; t < n; t += static_cast<long>(gridDim.x) * 256) {
        const int g = static_cast<int>(t % G);
        long r = t / G;
        const int x = static_cast<int>(r % W);
        r /= W;
        const int yv = static_cast<int>(r % H);
        const long b = r / H;
        const short8_t d = *reinterpret_cast<const short8_t*>(dy + ((b * (H / 2) + yv / 2) * (W / 2) + x / 2) * C + 8 * g);
        const short8_t s = *reinterpret_cast<const short8_t*>(skip + t * 8);
        short8_t v;
#pragma unroll
        for (int e = 0; e < 8; ++e)
            v[e] = static_cast<short>(f2bf(0.25f * bf2f(static_cast<bf16>(d[e])) + bf2f(static_cast<bf16>(s[e]))));
        *reinterpret_cast<short8_t*>(out + t * 8) = relu_masked(v, mask + t * 8);
    }
}

// Bilinear x2 (half-pixel centres, edge-clamped): output row Y samples input
// rows y0 = floor(Y / 2 - 1/4) and y0 + 1 with weights 3/4 and 1/4 (or 1/4 and
// 3/4), both clamped into [0, h - 1].
__device__ inline void up_taps(int Y, int h, int& a, int& b, float& wa, float& wb) {
    const int i = Y >> 1;
    if (Y & 1) {
        a = i;
        b = min(i + 1, h - 1);
        wa = 0.75f;
        wb = 0.25f;
    } else {
        a = max(i - 1, 0);
        b = i;
        wa = 0.25f;
        wb = 0.75f;
    }
}

// The decoder's input in one pass: y[p] = (bilinear x2 of x at p -- up_taps'
// two rows and two columns, wy_a (wx_a A + wx_b B) + wy_b (wx_a C + wx_b D) in
// FP32, rounded to bfloat16 -- channels [0, Ca); skip[p], channels [Ca, Ca + Cb)).
// One thread per (pixel, 8-channel group) with 16-byte loads and stores; Ca and
// Cb are multiples of 8.
__global__ __launch_bounds__(256) void k_upcat(const bf16* __restrict__ x, const bf16* __restrict__ skip,
                                              bf16* __restrict__ y, int N, int h, int w, int Ca, int Cb) {
    const int H = 2 * h, W = 2 * w, C = Ca + Cb, G = C / 8;
    const long n = static_cast<long>(N) * H * W * G;
    for (long t = static_cast<long>(blockIdx.x) * 256 + threadIdx.x; t < n; t += static_cast<long>(gridDim.x) * 256) {
        const int g = static_cast<int>(t % G);
        const long p = t / G;
        short8_t out;
        if (8 * g < Ca) {
            const int X = static_cast<int>(p % W);
            const long r = p / W;
            const int Y = static_cast<int>(r % H);
            const long b = r / H;
            int ya, yb, xa, xb;
            float wya, wyb, wxa, wxb;
            up_taps(Y, h, ya, yb, wya, wyb);
            up_taps(X, w, xa, xb, wxa, wxb);
            const bf16* q = x + b * h * w * Ca + 8 * g;
            const short8_t A = *reinterpret_cast<const short8_t*>(q + (static_cast<long>(ya) * w + xa) * Ca);
            const short8_t B = *reinterpret_cast<const short8_t*>(q + (static_cast<long>(ya) * w + xb) * Ca);
            const short8_t Cc = *reinterpret_cast<const short8_t*>(q + (static_cast<long>(yb) * w + xa) * Ca);
            const short8_t D = *reinterpret_cast<const short8_t*>(q + (static_cast<long>(yb) * w + xb) * Ca);
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const float v = wya * (wxa * bf2f(static_cast<bf16>(A[e])) + wxb * bf2f(static_cast<bf16>(B[e]))) +
                                wyb * (wxa * bf2f(static_cast<bf16>(Cc[e])) + wxb * bf2f(static_cast<bf16>(D[e])));
                out[e] = static_cast<short>(f2bf(v));
            }
        } else {
            out = *reinterpret_cast<const short8_t*>(skip + p * Cb + 8 * g - Ca);
        }
        *reinterpret_cast<short8_t*>(y + p * C + 8 * g) = out;
    }
}

// Its backward as a gather: input cell (i, j) collects every output cell whose
// taps include it (output rows 2i-2 .. 2i+3 cover all clamped cases), then the
// derivative of the ReLU that made the input (its output is mask).
__global__ __launch_bounds__(256) void k_upsample2_bwd(const bf16* __restrict__ dy, const bf16* __restrict__ mask,
                                                      bf16* __restrict__ dx, int N, int h, int w, int C) {
    const int H = 2 * h, W = 2 * w, G = C / 8;
    const long n = static_cast<long>(N) * h * w * G;
    for (long t = static_cast<long>(blockIdx.x) * 256 + threadIdx.x; t < n; t += static_cast<long>(gridDim.x) * 256) {
        const int g = static_cast<int>(t % G);
        long r = t / G;
        const int j = static_cast<int>(r % w);
        r /= w;
        const int i = static_cast<int>(r % h);
        const long b = r / h;
        float s[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
        for (int Y = max(2 * i - 2, 0); Y <= min(2 * i + 3, H - 1); ++Y) {
            int ya, yb;
            float wya, wyb;
            up_taps(Y, h, ya, yb, wya, wyb);
            const float wy = (ya == i ? wya : 0.f) + (yb == i ? wyb : 0.f);
            if (wy == 0.f) continue;
            for (int X = max(2 * j - 2, 0); X <= min(2 * j + 3, W - 1); ++X) {
                int xa, xb;
                float wxa, wxb;
                up_taps(X, w, xa, xb, wxa, wxb);
                const float wx = (xa == j ? wxa : 0.f) + (xb == j ? wxb : 0.f);
                if (wx == 0.f) continue;
                const short8_t d = *reinterpret_cast<const short8_t*>(dy + ((b * H + Y) * W + X) * C + 8 * g);
#pragma unroll
                for (int e = 0; e < 8; ++e) s[e] += wy * wx * bf2f(static_cast<bf16>(d[e]));
            }
        }
        short8_t v;
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = static_cast<short>(f2bf(s[e]));
        *reinterpret_cast<short8_t*>(dx + t * 8) = relu_masked(v, mask + t * 8);
    }
}

// Loss of the normalised prediction pred = o[p] + prev[p] against target[p]:
// sum of squares into *loss (one atomic per block), and the gradient of the
// mean, 2 (pred - target) / npix, into channel 0 of dout (16 channels).
__global__ __launch_bounds__(256) void k_mse(const float* __restrict__ o, const float* __restrict__ prev,
                                            const float* __restrict__ target, long npix, bf16* __restrict__ dout,
                                            float* __restrict__ loss) {
    __shared__ float part[4];
    float s = 0.f;
    const short8_t zero = {0, 0, 0, 0, 0, 0, 0, 0};
    for (long p = static_cast<long>(blockIdx.x) * 256 + threadIdx.x; p < npix; p += static_cast<long>(gridDim.x) * 256) {
        const float d = (o[p] + prev[p]) - target[p];
        s += d * d;
        short8_t v = zero;
        v[0] = static_cast<short>(f2bf(2.f * d / static_cast<float>(npix)));
        *reinterpret_cast<short8_t*>(dout + p * 16) = v;
        *reinterpret_cast<short8_t*>(dout + p * 16 + 8) = zero;
    }
    for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off);
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) atomicAdd(loss, (part[0] + part[1]) + (part[2] + part[3]));
}

// Every layer's gradients from its splits' partial sums, and Adam (Kingma and
// Ba 2015) on the fp32 masters, in one launch over all parameters; refreshes the
// bf16 weights w16 and the data gradient's, wt16[8 - tap][ci][co] = w[tap][co][ci].
// A block takes 64 neighbouring parameters; its 16 waves take every 16th split.
struct LayerSpan {
    long begin, wn, part;  // first parameter, weights (the biases follow), first partial sum
    int splits, cin, cout;
    bf16 *w16, *wt16;
};
template <int NL>
struct LayerSpans {
    LayerSpan l[NL];
};

template <int NL>
__global__ __launch_bounds__(1024) void k_reduce_adam(LayerSpans<NL> S, const float* __restrict__ part, long total,
                                                     float* __restrict__ w, float* __restrict__ g,
                                                     float* __restrict__ m, float* __restrict__ v, float lr, float b1,
                                                     float b2, float eps, float c1, float c2) {
    __shared__ float sums[16][64];
    const int lane = threadIdx.x & 63, slice = threadIdx.x >> 6;
    const long t = static_cast<long>(blockIdx.x) * 64 + lane;
    int k = 0;
    while (k + 1 < NL && t >= S.l[k + 1].begin) ++k;
    const LayerSpan L = S.l[k];
    const long q = t - L.begin, count = L.wn + L.cout;
    if (t < total) {
        const float* p = part + L.part + q;
        float s = 0.f;
#pragma unroll 8
        for (int i = slice; i < L.splits; i += 16) s += p[i * count];
        sums[slice][lane] = s;
    }
    __syncthreads();
    if (slice || t >= total) return;
    float gt = 0.f;
#pragma unroll
    for (int i = 0; i < 16; ++i) gt += sums[i][lane];
    g[t] = gt;
    const float mt = b1 * m[t] + (1.f - b1) * gt;
    const float vt = b2 * v[t] + (1.f - b2) * gt * gt;
    m[t] = mt;
    v[t] = vt;
    const float wn = w[t] - lr * (mt / c1) / (sqrtf(vt / c2) + eps);
    w[t] = wn;
    if (q < L.wn) {
        const bf16 r = f2bf(wn);
        const int ci = static_cast<int>(q % L.cin), co = static_cast<int>(q / L.cin % L.cout);
        const int tap = static_cast<int>(q / L.cin / L.cout);
        L.w16[q] = r;
        L.wt16[(static_cast<long>(8 - tap) * L.cin + ci) * L.cout + co] = r;
    }
}

// Host samples on the device: sums of squares of prev and d, per sample, in
// FP64 (blocks (N, G), as N may pass the grid's second dimension: partial sums [n][G][2]) ...
__global__ __launch_bounds__(256) void k_sumsq_samples(const float* __restrict__ d, const float* __restrict__ prev,
                                                      long hw, double* __restrict__ part) {
    const float4_t* a = reinterpret_cast<const float4_t*>(d + blockIdx.x * hw);
    const float4_t* b = reinterpret_cast<const float4_t*>(prev + blockIdx.x * hw);
    double sd = 0, sp = 0;
    for (long t = static_cast<long>(blockIdx.y) * 256 + threadIdx.x; t < hw / 4; t += static_cast<long>(gridDim.y) * 256) {
        const float4_t x = a[t], y = b[t];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            sd += static_cast<double>(x[i]) * x[i];
            sp += static_cast<double>(y[i]) * y[i];
        }
    }
    for (int off = 32; off > 0; off >>= 1) {
        sd += __shfl_xor(sd, off);
        sp += __shfl_xor(sp, off);
    }
    __shared__ double w[2][4];
    if ((threadIdx.x & 63) == 0) {
        w[0][threadIdx.x >> 6] = sp;
        w[1][threadIdx.x >> 6] = sd;
    }
    __syncthreads();
    if (threadIdx.x < 2)
        part[(static_cast<long>(blockIdx.x) * gridDim.y + blockIdx.y) * 2 + threadIdx.x] =
            (w[threadIdx.x][0] + w[threadIdx.x][1]) + (w[threadIdx.x][2] + w[threadIdx.x][3]);
}

// ... their scale s (the RMS of prev, else of d, else 1) and its inverse, one wave a sample ...
__global__ __launch_bounds__(64) void k_scale_samples(const double* __restrict__ part, int G, long hw,
                                                     float* __restrict__ scale, float* __restrict__ inv) {
    const double* p = part + static_cast<long>(blockIdx.x) * G * 2;
    double sp = 0, sd = 0;
    for (int k = threadIdx.x; k < G; k += 64) {
        sp += p[2 * k];
        sd += p[2 * k + 1];
    }
    for (int off = 32; off > 0; off >>= 1) {
        sp += __shfl_xor(sp, off);
        sd += __shfl_xor(sd, off);
    }
    if (threadIdx.x == 0) {
        double s = sqrt(sp / hw);
        if (!(s > 0)) s = sqrt(sd / hw);
        if (!(s > 0)) s = 1.0;
        scale[blockIdx.x] = static_cast<float>(s);
        inv[blockIdx.x] = static_cast<float>(1.0 / s);
    }
}

// ... and the network's input x0 = (d / s, prev / s, 0 ...) in bf16, with prev / s
// and target / s (target may be null; prev and target may be written in place).
__global__ __launch_bounds__(256) void k_pack_samples(const float* __restrict__ d, const float* prev, const float* target,
                                                     long hw, long npix, const float* __restrict__ inv,
                                                     bf16* __restrict__ x0, float* pv, float* tg) {
    const short8_t zero = {0, 0, 0, 0, 0, 0, 0, 0};
    for (long p = static_cast<long>(blockIdx.x) * 256 + threadIdx.x; p < npix; p += static_cast<long>(gridDim.x) * 256) {
        const float s = inv[p / hw];
        const float q = prev[p] * s;
        short8_t v = zero;
        v[0] = static_cast<short>(f2bf(d[p] * s));
        v[1] = static_cast<short>(f2bf(q));
        *reinterpret_cast<short8_t*>(x0 + p * 16) = v;
        *reinterpret_cast<short8_t*>(x0 + p * 16 + 8) = zero;
        pv[p] = q;
        if (target) tg[p] = target[p] * s;
    }
}

// out = (o + prev / s) * s
__global__ __launch_bounds__(256) void k_unpack_samples(const float* __restrict__ o, const float* __restrict__ pv,
                                                       const float* __restrict__ scale, long hw, long npix,
                                                       float* __restrict__ out) {
    for (long p = static_cast<long>(blockIdx.x) * 256 + threadIdx.x; p < npix; p += static_cast<long>(gridDim.x) * 256)
        out[p] = (o[p] + pv[p]) * scale[p / hw];
}

__global__ __launch_bounds__(256) void k_to_bf16(const float* __restrict__ a, bf16* __restrict__ b, long n) {
    for (long t = static_cast<long>(blockIdx.x) * 256 + threadIdx.x; t < n; t += static_cast<long>(gridDim.x) * 256)
        b[t] = f2bf(a[t]);
}

__global__ __launch_bounds__(256) void k_zero_f32(float* __restrict__ a, long n) {
    for (long t = static_cast<long>(blockIdx.x) * 256 + threadIdx.x; t < n; t += static_cast<long>(gridDim.x) * 256)
        a[t] = 0.f;
}

}  // namespace cnn
}  // namespace fs2d
