// unet.hip -- learned initial guess for the multigrid Poisson demag.
//
// A 2-D U-Net maps (m_x, m_y, m_z, film mask) on the plane of the MG box to
// the box potential, one output channel per z plane of the box.  Weights and
// activations are bf16 on the matrix cores (v_mfma_f32_16x16x32_bf16, FP32
// accumulation); gradients, master weights and Adam moments are FP32.  All of
// training runs here: forward, backward (data and weight gradients as
// implicit GEMMs), loss and optimiser.  The multigrid solver still decides
// convergence: the prediction only replaces the initial phi, and the solve
// iterates to the same residual (the reference has no counterpart; its solver starts from
// zero or from the previous solve, demag_poisson_mg.rs:1947-2057).
//
// Layout: activations channels-last, pixel p = (b*H + y)*W + x for batch b,
// row y, column x, every tensor dense.  Convolution weights [tap][c_out][c_in] with tap = (dy+1)*3+(dx+1),
// zero padding at the image border.
//
// Architecture (levels l = 0..3, c_l = base * 2^l):
//   enc_l: conv3x3(c_{l-1} or c_in -> c_l) + ReLU, conv3x3(c_l -> c_l) + ReLU,
//          2x2 average pool between levels;
//   dec_l (l = 2..0): nearest 2x upsample of the level below, concatenated
//          [up, skip] with enc_l's output, then two conv3x3 + ReLU to c_l;
//   head:  conv3x3(c_0 -> c_out), linear, FP32 output.
#include "../../include/llgmi.h"
#include "common.hpp"

#include <cmath>
#include <cstdlib>
#include <cstring>
#include <memory>
#include <mutex>
#include <set>
#include <string>
#include <type_traits>
#include <vector>

namespace llgmi {
namespace {

typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kLevels = 4;
constexpr int kNT = 256;

__device__ __forceinline__ uint16_t f2bf(float f) {   // round to nearest even
    uint32_t u = __float_as_uint(f);
    u += 0x7fffu + ((u >> 16) & 1u);
    return (uint16_t)(u >> 16);
}
__device__ __forceinline__ float bf2f(uint16_t h) { return __uint_as_float((uint32_t)h << 16); }


// Input of a convolution, channels last: channels [0, lo_c) are the nearest 2x
// upsampling of a half-resolution tensor (dense lo_c channels, lo_c a multiple
// of 32), the rest come from a dense tensor of hi_c channels at the output's
// resolution.  So a decoder's concatenation [up, skip] is never stored.
struct ConvSrc {
    const uint16_t *lo;
    int lo_c;
    const uint16_t *hi;
    int hi_c;
};
// The value, hidden from the optimiser: addresses formed from it are recomputed
// where they are used instead of being kept in registers over a block's loops.
__device__ __forceinline__ int opaque(int v) {
    asm volatile("" : "+v"(v));
    return v;
}
// the 8 channels from c on of pixel (b, yy, xx), zero outside the image
__device__ __forceinline__ uint4 src_load(const ConvSrc &s, int c, bool low, int b, int yy, int xx, int H, int W) {
    if (yy < 0 || yy >= H || xx < 0 || xx >= W) return uint4{0u, 0u, 0u, 0u};
    const uint16_t *p = low ? s.lo + ((int64_t)(b * (H >> 1) + (yy >> 1)) * (W >> 1) + (xx >> 1)) * s.lo_c + c
                            : s.hi + ((int64_t)(b * H + yy) * W + xx) * s.hi_c + (c - s.lo_c);
    return *reinterpret_cast<const uint4 *>(p);
}

// What a convolution does with its sums (in FP32 registers):
//  ACT   bf16 of relu(sum + bias) to y; with pool also its 2x2 average
//  F32   sum (+ bias) to yf
//  MASK  bf16 of the sum where mask > 0, else 0, to y: a data gradient and the
//        ReLU backward of the layer before it
//  MSE   the loss's terms of sum + bias against tgt (channels < cv, pixels
//        x < wv <= W, y < hv <= H: a tile overhangs the image) added to *loss, and
//        the bf16 of the loss gradient to y
//  CAT   data gradient of a concatenation [up, skip]: channels < up_c are summed
//        over 2x2 pixels (the upsampling's gradient) and masked into y at half
//        resolution, the rest go to yf in FP32
enum { EPI_ACT, EPI_F32, EPI_MASK, EPI_MSE, EPI_CAT };
struct ConvEpi {
    uint16_t *y = nullptr;
    float *yf = nullptr;
    uint16_t *pool = nullptr;
    const uint16_t *mask = nullptr;
    int up_c = 0;
    const uint16_t *tgt = nullptr;
    int cv = 0, wv = 0, hv = 0;
    double inv_count = 0.0;
    double *loss = nullptr;
};

__device__ __forceinline__ uint4 relu_mask(uint4 v, uint4 m) {
    uint16_t *hv = reinterpret_cast<uint16_t *>(&v);
    const uint16_t *hm = reinterpret_cast<const uint16_t *>(&m);
#pragma unroll
    for (int k = 0; k < 8; ++k)
        if (!(bf2f(hm[k]) > 0.f)) hv[k] = 0;
    return v;
}

// 3x3 convolution as an implicit GEMM on gfx950's K = 32 bf16 matrix-core
// product: rows = pixels, columns = output channels, reduction = 9 taps x input
// channels.  Also the data gradient (the output gradient with tap-flipped,
// transposed weights).  A block computes TH x 16*TW pixels for 16*NT output
// channels; wave w owns TH/4 pixel rows.  Input channels go in chunks of 32: a
// chunk's haloed input tile and its weights of all nine taps are staged in LDS
// through registers, the next chunk's loads in flight during the products.
//
// LDS reads bound a straightforward loop over taps (one input operand per
// product pair), so the nine taps' weights are held in registers and the
// wave walks the input rows once: input row i serves output rows i, i-1, i-2
// (taps dy = 0, 1, 2), a third of the reads.  Per chunk and wave of the 16 x 32
// tile: 54 KB of LDS reads for 144 products, 93 of the CU's 128 bytes per clock
// at the matrix cores' full rate.  Every sum still takes its chunks in order and
// within a chunk its taps 0..8.
//
// The sums leave through LDS as whole 16-byte pieces of a pixel (two-byte stores
// of the product's own layout took as long as the products), with the pass that
// would follow (pooling, upsampling, the ReLU's gradient, the loss) applied on
// the way out.  A layer of one chunk keeps its weights in LDS over a block's run
// of tiles.
// Requires cin % 16 == 0, cout % (16*NT) == 0; H, W even for pool and CAT.
// Measured against the tap-by-tap tile kernel with separate pooling, upsampling,
// concatenation, ReLU-gradient and loss passes: forward at 528 x 528 467 -> 365
// us, training step at batch 8 8.10 -> 5.84 ms; with the loss's targets through
// LDS, three blocks per CU for the 16-wide tiles and even runs of tiles 333 us and
// 5.59 ms.
constexpr int kKC = 32, kKRow = kKC + 8;   // channel chunk; LDS row, padded against bank conflicts
template <int TH, int TW, int NT>
struct ConvShape {
    static constexpr int CO = 16 * NT, XW = 16 * TW + 2, NPX = (TH + 2) * XW, NOUT = TH * 16 * TW;
    static constexpr int kXin = NPX * kKRow, kOut = NOUT * (CO + 8), kReg = kXin > kOut ? kXin : kOut;
    static constexpr size_t LDS = sizeof(uint16_t) * (size_t)(kReg + 9 * CO * kKRow);
};
// blocks per CU a tile's registers and LDS allow
template <int TW, int NT>
constexpr int conv_blocks_per_cu() { return TW == 1 && NT < 3 ? 3 : 2; }
template <int TH, int TW, int NT, int EPI, bool RELU>
__global__ __launch_bounds__(256, (conv_blocks_per_cu<TW, NT>())) void k_conv3x3(ConvSrc src, int cin, const uint16_t *__restrict__ w,
                                                    const float *__restrict__ bias, ConvEpi ep, int cout, int B,
                                                    int H, int W) {
    using S = ConvShape<TH, TW, NT>;
    constexpr int RW = TH / 4, CO = S::CO, XW = S::XW, NPX = S::NPX, OROW = CO + 8;
    extern __shared__ __align__(16) unsigned char conv_smem[];
    uint16_t *xin = reinterpret_cast<uint16_t *>(conv_smem);   // [NPX][kKRow], later the output tile [pixel][OROW]
    uint16_t *wl = xin + S::kReg;                              // [9][CO][kKRow]
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, li = lane & 15, g = lane >> 4;
    const int ntx = (W + 16 * TW - 1) / (16 * TW), nty = (H + TH - 1) / TH, ntile = ntx * nty * B;
    const int t0 = (int)((int64_t)ntile * blockIdx.x / gridDim.x),
              t1 = (int)((int64_t)ntile * (blockIdx.x + 1) / gridDim.x);
    const int co_base = (int)blockIdx.y * CO;
    const bool one_chunk = cin <= kKC;
    constexpr int NI = (NPX * 4 + 255) / 256, NW = (9 * CO * 4 + 255) / 256;
    uint4 ri[NI], rw[NW];
    auto fetch_x = [&](int t, int c0) {
        const int x0 = (t % ntx) * 16 * TW, y0 = ((t / ntx) % nty) * TH, b = t / (ntx * nty);
        const bool low = c0 < src.lo_c;
        const int tid = opaque(threadIdx.x);
#pragma unroll
        for (int k = 0; k < NI; ++k) {
            const int e = tid + k * 256, pix = e >> 2, c = c0 + (e & 3) * 8;
            ri[k] = uint4{0u, 0u, 0u, 0u};
            if (e < NPX * 4 && c < cin) ri[k] = src_load(src, c, low, b, y0 + pix / XW - 1, x0 + pix % XW - 1, H, W);
        }
    };
    auto fetch_w = [&](int c0) {
        const int tid = opaque(threadIdx.x);
#pragma unroll
        for (int k = 0; k < NW; ++k) {
            const int e = tid + k * 256, row = e >> 2, c = c0 + (e & 3) * 8;   // row = tap * CO + co
            const int tap = row / CO, co = row - tap * CO;
            rw[k] = uint4{0u, 0u, 0u, 0u};
            if (e < 9 * CO * 4 && c < cin)
                rw[k] = *reinterpret_cast<const uint4 *>(w + ((int64_t)tap * cout + co_base + co) * cin + c);
        }
    };
    double lsum = 0.0;
    if (t0 < t1) {
        fetch_x(t0, 0);
        fetch_w(0);
    }
    for (int t = t0; t < t1; ++t) {
        const int x0 = (t % ntx) * 16 * TW, y0 = ((t / ntx) % nty) * TH, b = t / (ntx * nty);
        f32x4 acc[RW][TW][NT];
#pragma unroll
        for (int r = 0; r < RW; ++r)
#pragma unroll
            for (int h = 0; h < TW; ++h)
#pragma unroll
                for (int nt = 0; nt < NT; ++nt) acc[r][h][nt] = f32x4{0.f, 0.f, 0.f, 0.f};
        for (int c0 = 0; c0 < cin; c0 += kKC) {
            __syncthreads();   // the previous chunk's (or output tile's) reads are done
#pragma unroll
            for (int k = 0; k < NI; ++k) {
                const int e = threadIdx.x + k * 256;
                if (e < NPX * 4) *reinterpret_cast<uint4 *>(xin + (e >> 2) * kKRow + (e & 3) * 8) = ri[k];
            }
            if (!one_chunk || t == t0) {
#pragma unroll
                for (int k = 0; k < NW; ++k) {
                    const int e = threadIdx.x + k * 256;
                    if (e < 9 * CO * 4) *reinterpret_cast<uint4 *>(wl + (e >> 2) * kKRow + (e & 3) * 8) = rw[k];
                }
            }
            __syncthreads();
            if (c0 + kKC < cin) {
                fetch_x(t, c0 + kKC);
                fetch_w(c0 + kKC);
            } else if (t + 1 < t1) {
                fetch_x(t + 1, 0);
                if (!one_chunk) fetch_w(0);
            }
            bf16x8 bw[9][NT];
#pragma unroll
            for (int tap = 0; tap < 9; ++tap)
#pragma unroll
                for (int nt = 0; nt < NT; ++nt)
                    bw[tap][nt] = *reinterpret_cast<const bf16x8 *>(wl + (tap * CO + nt * 16 + li) * kKRow + g * 8);
#pragma unroll
            for (int i = 0; i < RW + 2; ++i) {
                bf16x8 a[3][TW];
#pragma unroll
                for (int dx = 0; dx < 3; ++dx)
#pragma unroll
                    for (int h = 0; h < TW; ++h)
                        a[dx][h] = *reinterpret_cast<const bf16x8 *>(
                            xin + ((wave * RW + i) * XW + h * 16 + li + dx) * kKRow + g * 8);
#pragma unroll
                for (int dy = 0; dy < 3; ++dy) {
                    const int r = i - dy;
                    if (r < 0 || r >= RW) continue;
#pragma unroll
                    for (int dx = 0; dx < 3; ++dx)
#pragma unroll
                        for (int h = 0; h < TW; ++h)
#pragma unroll
                            for (int nt = 0; nt < NT; ++nt)
                                acc[r][h][nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                                    a[dx][h], bw[dy * 3 + dx][nt], acc[r][h][nt], 0, 0, 0);
                }
            }
        }
        // lane holds pixels 4 g + q of each 16-pixel tile, channel li
        const bool cat_up = EPI == EPI_CAT && co_base < ep.up_c;
        if (EPI == EPI_F32 || (EPI == EPI_CAT && !cat_up)) {
            const int cs = EPI == EPI_CAT ? cout - ep.up_c : cout, cb = EPI == EPI_CAT ? co_base - ep.up_c : co_base;
#pragma unroll
            for (int r = 0; r < RW; ++r) {
                const int yy = y0 + wave * RW + r;
                if (yy >= H) continue;
#pragma unroll
                for (int h = 0; h < TW; ++h)
#pragma unroll
                    for (int nt = 0; nt < NT; ++nt) {
                        const int co = nt * 16 + li;
                        const float bv = bias ? bias[co_base + co] : 0.f;
#pragma unroll
                        for (int q = 0; q < 4; ++q) {
                            const int xx = x0 + h * 16 + g * 4 + q;
                            if (xx < W) ep.yf[((int64_t)(b * H + yy) * W + xx) * cs + cb + co] = acc[r][h][nt][q] + bv;
                        }
                    }
            }
            continue;
        }
        __syncthreads();   // every wave's reads of xin are done
        if constexpr (EPI == EPI_MSE) {
            // the tile's targets into the places their gradients will take, in
            // 16-byte pieces (read in the products' layout, two bytes a lane, they
            // took longer than the convolution); the caller's buffer may start on any
            // element
            const int tid = opaque(threadIdx.x);
            auto targets = [&](auto load) {
                for (int e = tid; e < TH * 16 * TW * (CO / 8); e += 256) {
                    const int px = e / (CO / 8), c = (e % (CO / 8)) * 8;
                    const int yy = y0 + px / (16 * TW), xx = x0 + px % (16 * TW);
                    uint4 tv{0u, 0u, 0u, 0u};
                    if (yy < H && xx < W) tv = load(ep.tgt + ((int64_t)(b * H + yy) * W + xx) * cout + co_base + c);
                    *reinterpret_cast<uint4 *>(xin + px * OROW + c) = tv;
                }
            };
            if ((reinterpret_cast<uintptr_t>(ep.tgt) & 15) == 0) {
                targets([](const uint16_t *p) { return *reinterpret_cast<const uint4 *>(p); });
            } else {
                targets([](const uint16_t *p) {
                    uint4 tv;
                    uint16_t *h = reinterpret_cast<uint16_t *>(&tv);
#pragma unroll
                    for (int k = 0; k < 8; ++k) h[k] = p[k];
                    return tv;
                });
            }
            __syncthreads();
        }
        if (cat_up) {
            if constexpr (EPI == EPI_CAT) {
#pragma unroll
                for (int r = 0; r < RW; r += 2)
#pragma unroll
                    for (int h = 0; h < TW; ++h)
#pragma unroll
                        for (int nt = 0; nt < NT; ++nt)
#pragma unroll
                            for (int q = 0; q < 4; q += 2) {
                                const float v = acc[r][h][nt][q] + acc[r][h][nt][q + 1] + acc[r + 1][h][nt][q] +
                                                acc[r + 1][h][nt][q + 1];
                                const int px = ((wave * RW + r) / 2) * 8 * TW + h * 8 + (g * 4 + q) / 2;
                                xin[px * OROW + nt * 16 + li] = f2bf(v);
                            }
            }
        } else {
#pragma unroll
            for (int r = 0; r < RW; ++r)
#pragma unroll
                for (int h = 0; h < TW; ++h)
#pragma unroll
                    for (int nt = 0; nt < NT; ++nt) {
                        const int co = co_base + nt * 16 + li;
                        const float bv = bias ? bias[co] : 0.f;
#pragma unroll
                        for (int q = 0; q < 4; ++q) {
                            float v = acc[r][h][nt][q] + bv;
                            if (RELU) v = fmaxf(v, 0.f);
                            uint16_t &at = xin[((wave * RW + r) * 16 * TW + h * 16 + g * 4 + q) * OROW + nt * 16 + li];
                            if constexpr (EPI == EPI_MSE) {
                                const int yy = y0 + wave * RW + r, xx = x0 + h * 16 + g * 4 + q;
                                float gr = 0.f;
                                if (co < ep.cv && xx < ep.wv && yy < ep.hv) {
                                    const double d = (double)v - (double)bf2f(at);
                                    lsum += d * d;
                                    gr = (float)(2.0 * d * ep.inv_count);
                                }
                                v = gr;
                            }
                            at = f2bf(v);
                        }
                    }
        }
        __syncthreads();
        // out of LDS in 16-byte pieces (8 channels of a pixel)
        const int tid = opaque(threadIdx.x);
        const int sh = cat_up ? 1 : 0;   // CAT: half resolution
        const int Ho = H >> sh, Wo = W >> sh, co_n = cat_up ? ep.up_c : cout, ow = (16 * TW) >> sh;
        constexpr int P8 = CO / 8;
        for (int e = tid; e < ((TH * 16 * TW) >> (2 * sh)) * P8; e += 256) {
            const int px = e / P8, c = (e % P8) * 8;
            const int yy = (y0 >> sh) + px / ow, xx = (x0 >> sh) + px % ow;
            if (yy >= Ho || xx >= Wo) continue;
            uint4 v = *reinterpret_cast<const uint4 *>(xin + px * OROW + c);
            const int64_t o = ((int64_t)(b * Ho + yy) * Wo + xx) * co_n + co_base + c;
            if (EPI == EPI_MASK || EPI == EPI_CAT) v = relu_mask(v, *reinterpret_cast<const uint4 *>(ep.mask + o));
            *reinterpret_cast<uint4 *>(ep.y + o) = v;
        }
        if (EPI == EPI_ACT && ep.pool) {
            for (int e = tid; e < (TH / 2 * 8 * TW) * P8; e += 256) {
                const int px = e / P8, c = (e % P8) * 8, py = px / (8 * TW), pxx = px % (8 * TW);
                const int yy = (y0 >> 1) + py, xx = (x0 >> 1) + pxx;
                if (yy >= (H >> 1) || xx >= (W >> 1)) continue;
                const uint16_t *q0 = xin + (2 * py * 16 * TW + 2 * pxx) * OROW + c;
                const uint16_t *q1 = q0 + OROW, *q2 = q0 + 16 * TW * OROW, *q3 = q2 + OROW;
                uint4 o;
                uint16_t *ho = reinterpret_cast<uint16_t *>(&o);
#pragma unroll
                for (int k = 0; k < 8; ++k)
                    ho[k] = f2bf(0.25f * (bf2f(q0[k]) + bf2f(q1[k]) + bf2f(q2[k]) + bf2f(q3[k])));
                *reinterpret_cast<uint4 *>(ep.pool + ((int64_t)(b * (H >> 1) + yy) * (W >> 1) + xx) * cout + co_base + c) = o;
            }
        }
    }
    if constexpr (EPI == EPI_MSE) {
        __shared__ double lpart[4];
        for (int o = 32; o > 0; o >>= 1) lsum += __shfl_xor(lsum, o);
        if (lane == 0) lpart[wave] = lsum;
        __syncthreads();
        if (threadIdx.x == 0) atomicAdd(ep.loss, (lpart[0] + lpart[1] + lpart[2] + lpart[3]) * ep.inv_count);
    }
}

// Weight and bias gradient: dw[tap][co][ci] = sum_p dz[p][co] x[p + off(tap)][ci],
// db[co] = sum_p dz[p][co].  The reduction runs over pixels, which a matrix-core
// operand wants eight at a time per channel while memory holds channels
// together: the tiles are staged in LDS as they lie in memory ([pixel][channel])
// and read with the transposing LDS read (ds_read_b64_tr_b16, four pixels of
// one channel per lane), so a tap is an address offset and needs no copy of its
// own.  A block takes one (16*MT) x (16*NT) channel tile and a contiguous run
// of 16 x 16 pixel tiles: per tile dz and x with its one-pixel halo are loaded
// once (the next tile's loads are in flight during the products) and serve all
// nine taps, whose 9*MT*NT partial tiles stay in registers until the run ends.
// Each wave takes four pixel rows (two K = 32 products of two 16-pixel rows);
// the waves' sums are added through LDS and written to the block's own row of
// `part`, which k_part_sum reduces: no atomics, so gradients do not depend on
// the order in which blocks finish.  The bias gradient is one more product,
// with ones, in the blocks of the first ci tile.
// Bound by the tiles' loads where a layer has few channels (32 x 32: 72
// multiply-adds per byte) and by LDS reads elsewhere.  Against one block per tap
// with 8-byte loads and atomics (and a pass of its own for the bias): 11.3 -> 1.3 ms for the fifteen layers of a
// 8 x 528 x 528 step (742 -> 84 us per 32 x 32 tiled layer).
constexpr int kWgT = 16, kWgX = kWgT + 2;   // pixel tile and tile with halo
template <int MT, int NT>
__global__ __launch_bounds__(256, 2) void k_conv3x3_wgrad(const uint16_t *__restrict__ dz, int cout, ConvSrc src,
                                                          int cin, float *__restrict__ part, int B, int H, int W) {
    constexpr int CO = 16 * MT, CI = 16 * NT;
    constexpr int NX = kWgX * kWgX * (CI / 8), NZ = kWgT * kWgT * (CO / 8);   // 16-byte pieces of a tile
    constexpr int LX = (NX + 255) / 256, LZ = (NZ + 255) / 256;
    constexpr size_t kStage = 16 * (size_t)(NX + NZ), kRed = sizeof(f32x4) * 4 * MT * NT * 64;
    __shared__ __align__(16) unsigned char smem[kStage > kRed ? kStage : kRed];
    uint16_t *xin = reinterpret_cast<uint16_t *>(smem);      // [kWgX * kWgX][CI]
    uint16_t *zin = xin + kWgX * kWgX * CI;                  // [kWgT * kWgT][CO]
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, g = lane >> 4, j = lane & 15;
    const int co_tiles = cout / CO;
    const int co_base = ((int)blockIdx.y % co_tiles) * CO, ci_base = ((int)blockIdx.y / co_tiles) * CI;
    const int ntx = (W + kWgT - 1) / kWgT, nty = (H + kWgT - 1) / kWgT, ntile = ntx * nty * B;
    const int t0 = (int)((int64_t)ntile * blockIdx.x / gridDim.x),
              t1 = (int)((int64_t)ntile * (blockIdx.x + 1) / gridDim.x);
    f32x4 acc[9][MT][NT], accb[MT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
        accb[mt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int tap = 0; tap < 9; ++tap)
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) acc[tap][mt][nt] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    const bool low = ci_base < src.lo_c;
    uint4 rx[LX], rz[LZ];
    auto fetch = [&](int t) {
        const int tx = t % ntx, ty = (t / ntx) % nty, b = t / (ntx * nty);
        const int x0 = tx * kWgT, y0 = ty * kWgT;
#pragma unroll
        for (int k = 0; k < LX; ++k) {
            const int e = threadIdx.x + k * 256, pix = e / (CI / 8), c = (e % (CI / 8)) * 8;
            rx[k] = uint4{0u, 0u, 0u, 0u};
            if (e < NX)
                rx[k] = src_load(src, ci_base + c, low, b, y0 + pix / kWgX - 1, x0 + pix % kWgX - 1, H, W);
        }
#pragma unroll
        for (int k = 0; k < LZ; ++k) {
            const int e = threadIdx.x + k * 256, pix = e / (CO / 8), c = (e % (CO / 8)) * 8;
            const int yy = y0 + pix / kWgT, xx = x0 + pix % kWgT;
            rz[k] = uint4{0u, 0u, 0u, 0u};
            if (e < NZ && yy < H && xx < W)
                rz[k] = *reinterpret_cast<const uint4 *>(dz + ((int64_t)(b * H + yy) * W + xx) * cout + co_base + c);
        }
    };
    // eight pixels (k = 8 g + 0..7) of channel j of the 16 at p
    auto frag = [&](const uint16_t *p, int row_len) -> bf16x8 {
        typedef __attribute__((address_space(3))) bf16x4 *lds4;
        const bf16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds4)p);
        const bf16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds4)(p + 4 * row_len));
        typedef short s16x8 __attribute__((ext_vector_type(8)));
        return __builtin_bit_cast(bf16x8, (s16x8)__builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
    };
    const __bf16 one = (__bf16)1.0f;
    const bf16x8 ones = {one, one, one, one, one, one, one, one};
    if (t0 < t1) fetch(t0);
    for (int t = t0; t < t1; ++t) {
        __syncthreads();   // the previous tile's reads are done
#pragma unroll
        for (int k = 0; k < LX; ++k)
            if (threadIdx.x + k * 256 < NX) reinterpret_cast<uint4 *>(xin)[threadIdx.x + k * 256] = rx[k];
#pragma unroll
        for (int k = 0; k < LZ; ++k)
            if (threadIdx.x + k * 256 < NZ) reinterpret_cast<uint4 *>(zin)[threadIdx.x + k * 256] = rz[k];
        __syncthreads();
        if (t + 1 < t1) fetch(t + 1);
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            // lane group g: row g / 2 of the step's two, columns 8 (g % 2) ..
            const int row = (wave * 2 + s) * 2 + (g >> 1), col = (g & 1) * 8 + (j >> 2);
            const uint16_t *za = zin + (row * kWgT + col) * CO + (j & 3) * 4;
            const uint16_t *xa = xin + (row * kWgX + col) * CI + (j & 3) * 4;
            bf16x8 a[MT];
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) a[mt] = frag(za + mt * 16, CO);
            if (ci_base == 0) {
#pragma unroll
                for (int mt = 0; mt < MT; ++mt)
                    accb[mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[mt], ones, accb[mt], 0, 0, 0);
            }
#pragma unroll
            for (int tap = 0; tap < 9; ++tap) {
                bf16x8 bx[NT];
#pragma unroll
                for (int nt = 0; nt < NT; ++nt) bx[nt] = frag(xa + ((tap / 3) * kWgX + tap % 3) * CI + nt * 16, CI);
#pragma unroll
                for (int mt = 0; mt < MT; ++mt)
#pragma unroll
                    for (int nt = 0; nt < NT; ++nt)
                        acc[tap][mt][nt] =
                            __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[mt], bx[nt], acc[tap][mt][nt], 0, 0, 0);
            }
        }
    }
    // the four waves' sums through LDS, one tap at a time; lane holds rows
    // 4 (lane / 16) + r (co), column lane % 16 (ci) of every 16 x 16 tile
    f32x4(*red)[MT * NT][64] = reinterpret_cast<f32x4(*)[MT * NT][64]>(smem);
    float *out = part + (int64_t)blockIdx.x * ((int64_t)9 * cout * cin + cout);
#pragma unroll
    for (int tap = 0; tap < 9; ++tap) {
        __syncthreads();
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) red[wave][mt * NT + nt][lane] = acc[tap][mt][nt];
        __syncthreads();
        for (int e = threadIdx.x; e < MT * NT * 64; e += 256) {
            const int t = e / 64, ln = e % 64;
            const f32x4 sum = red[0][t][ln] + red[1][t][ln] + red[2][t][ln] + red[3][t][ln];
            const int ci = ci_base + (t % NT) * 16 + (ln & 15);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int co = co_base + (t / NT) * 16 + (ln >> 4) * 4 + r;
                out[((int64_t)tap * cout + co) * cin + ci] = sum[r];
            }
        }
    }
    if (ci_base == 0) {   // uniform over the block
        __syncthreads();
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) red[wave][mt][lane] = accb[mt];
        __syncthreads();
        for (int e = threadIdx.x; e < MT * 64; e += 256) {
            const int t = e / 64, ln = e % 64;
            if (ln & 15) continue;   // every column of the product with ones is the same sum
            const f32x4 sum = red[0][t][ln] + red[1][t][ln] + red[2][t][ln] + red[3][t][ln];
#pragma unroll
            for (int r = 0; r < 4; ++r) out[(int64_t)9 * cout * cin + co_base + t * 16 + (ln >> 4) * 4 + r] = sum[r];
        }
    }
}

// out[i] = sum of part[s][i] over the nrow rows of length n: four row groups of
// 64 columns per block, added through LDS
__global__ __launch_bounds__(256) void k_part_sum(const float *__restrict__ part, int nrow, int64_t n,
                                                  float *__restrict__ out) {
    __shared__ float red[4][64];
    const int c = threadIdx.x & 63, g = threadIdx.x >> 6;
    const int64_t i = (int64_t)blockIdx.x * 64 + c;
    float s = 0.f;
    if (i < n) {
#pragma unroll 8
        for (int r = g; r < nrow; r += 4) s += part[(int64_t)r * n + i];
    }
    red[g][c] = s;
    __syncthreads();
    if (g == 0 && i < n) out[i] = (red[0][c] + red[1][c]) + (red[2][c] + red[3][c]);
}

// Gradient of an encoder's output, eight channels per thread: its skip part
// plus a quarter of the pooled tensor's gradient, masked by the ReLU, as bf16:
// dz[fine][c] = bf16((gs[fine][c] + 0.25 gp[coarse][c]) where y > 0)
__global__ void k_skip_pool_relu(const float *__restrict__ gs, const float *__restrict__ gp,
                                 const uint16_t *__restrict__ y, int C, uint16_t *__restrict__ dz, int B, int H,
                                 int W) {
    const int C8 = C / 8;
    const int64_t n = (int64_t)B * H * W * C8;
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        const int c = (int)(i % C8) * 8;
        const int64_t p = i / C8;
        const int x = (int)(p % W), yy = (int)((p / W) % H), b = (int)(p / ((int64_t)W * H));
        const int64_t pc = ((int64_t)b * (H / 2) + yy / 2) * (W / 2) + x / 2;
        const float4 s0 = *reinterpret_cast<const float4 *>(gs + p * C + c),
                     s1 = *reinterpret_cast<const float4 *>(gs + p * C + c + 4),
                     q0 = *reinterpret_cast<const float4 *>(gp + pc * C + c),
                     q1 = *reinterpret_cast<const float4 *>(gp + pc * C + c + 4);
        const float v[8] = {s0.x + 0.25f * q0.x, s0.y + 0.25f * q0.y, s0.z + 0.25f * q0.z, s0.w + 0.25f * q0.w,
                            s1.x + 0.25f * q1.x, s1.y + 0.25f * q1.y, s1.z + 0.25f * q1.z, s1.w + 0.25f * q1.w};
        uint4 o;
        uint16_t *ho = reinterpret_cast<uint16_t *>(&o);
#pragma unroll
        for (int k = 0; k < 8; ++k) ho[k] = f2bf(v[k]);
        *reinterpret_cast<uint4 *>(dz + p * C + c) =
            relu_mask(o, *reinterpret_cast<const uint4 *>(y + p * C + c));
    }
}

// Adam (Kingma & Ba 2015) on FP32 master parameters; bc1 = 1 - b1^t, bc2 = 1 - b2^t
__global__ void k_adam(float *__restrict__ p, const float *__restrict__ g, float *__restrict__ m,
                       float *__restrict__ v, int64_t n, float lr, float b1, float b2, float eps, float bc1,
                       float bc2) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        const float gi = g[i];
        const float mi = b1 * m[i] + (1.f - b1) * gi;
        const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
        m[i] = mi;
        v[i] = vi;
        p[i] -= lr * (mi / bc1) / (sqrtf(vi / bc2) + eps);
    }
}

// bf16 weights of every convolution (blockIdx.y) for the forward product (same
// layout) and for the data gradient: wb[tap'][ci][co] = w[8 - tap'][co][ci].  One
// launch: a layer's cast is shorter than a launch.
constexpr int kConvs = 4 * kLevels - 1;
struct CastLayer {
    int64_t w_off;
    int cout, cin;
    uint16_t *wf, *wb;
};
struct CastLayers {
    CastLayer l[kConvs];
};
__global__ void k_w_cast(const float *__restrict__ p, CastLayers layers) {
    const CastLayer L = layers.l[blockIdx.y];
    const float *w = p + L.w_off;
    const int n = 9 * L.cout * L.cin;
    for (int i = (int)(blockIdx.x * blockDim.x + threadIdx.x); i < n; i += (int)(gridDim.x * blockDim.x)) {
        const int ci = i % L.cin, co = (i / L.cin) % L.cout, tap = i / (L.cin * L.cout);
        const uint16_t h = f2bf(w[i]);
        L.wf[i] = h;
        L.wb[((8 - tap) * L.cin + ci) * L.cout + co] = h;
    }
}

// Input packing: x[b][y][x][0..3] = (m_x, m_y, m_z, |m|^2 > 1e-30) of film
// cell (x - offx, y - offy), zero outside the film; channels 4..15 zero.
template <typename T>
__global__ void k_pack_input(const T *__restrict__ m, int nx, int ny, int offx, int offy, uint16_t *__restrict__ xo,
                             int H, int W) {
    const int64_t n = (int64_t)H * W;
    const int64_t nc = (int64_t)nx * ny;
    for (int64_t p = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; p < n; p += (int64_t)gridDim.x * blockDim.x) {
        const int x = (int)(p % W) - offx, y = (int)(p / W) - offy;
        float v[4] = {0.f, 0.f, 0.f, 0.f};
        if (x >= 0 && x < nx && y >= 0 && y < ny) {
            const int64_t c = (int64_t)y * nx + x;
            const double mx = m[c], my = m[nc + c], mz = m[2 * nc + c];
            v[0] = (float)mx;
            v[1] = (float)my;
            v[2] = (float)mz;
            v[3] = (mx * mx + my * my + mz * mz) > 1e-30 ? 1.f : 0.f;
        }
        uint16_t *o = xo + p * 16;
        for (int c = 0; c < 16; ++c) o[c] = c < 4 ? f2bf(v[c]) : (uint16_t)0;
    }
}

// box potential phi[z][y][x] (px x py x pz) -> target t[y][x][z] / scale
__global__ void k_pack_phi(const double *__restrict__ phi, int px, int py, int pz, double inv_scale,
                           uint16_t *__restrict__ t, int C, int H, int W) {
    const int64_t n = (int64_t)H * W * C;
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        const int c = (int)(i % C);
        const int64_t p = i / C;
        const int x = (int)(p % W), y = (int)(p / W);
        float v = 0.f;
        if (c < pz && x < px && y < py) v = (float)(phi[((int64_t)c * py + y) * px + x] * inv_scale);
        t[i] = f2bf(v);
    }
}

// network output y[y][x][z] (FP32) -> box potential phi[z][y][x] * scale
__global__ void k_unpack_phi(const float *__restrict__ yv, int C, int H, int W, double scale, int accumulate,
                             double *__restrict__ phi, int px, int py, int pz) {
    const int64_t n = (int64_t)px * py * pz;
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        const int x = (int)(i % px), y = (int)((i / px) % py), z = (int)(i / ((int64_t)px * py));
        const double v = (double)yv[((int64_t)y * W + x) * C + z] * scale;
        phi[i] = accumulate ? phi[i] + v : v;
    }
}

inline int grid_of(int64_t n) { return (int)std::min<int64_t>((n + kNT - 1) / kNT, 16384); }

}  // namespace

// ---------------------------------------------------------------------------
// Host side: the network, its buffers and one training step.
// ---------------------------------------------------------------------------
struct UNetConv {
    int cin = 0, cout = 0;
    bool relu = true;
    int64_t w_off = 0, b_off = 0;   // offsets in the FP32 parameter vector
    uint16_t *wf = nullptr, *wb = nullptr;
};

struct UNet {
    int B, H, W, cin_real, cout_real, cout, base, wv, hv;
    hipStream_t stream = nullptr;
    std::vector<UNetConv> conv;   // enc (2 per level), dec (2 per level 2..0), head
    int64_t nparam = 0;
    float *d_p = nullptr, *d_g = nullptr, *d_m = nullptr, *d_v = nullptr;
    uint16_t *d_wbf = nullptr;    // bf16 forward and transposed weights of every conv
    float *d_part = nullptr;      // partial weight gradients of one layer
    int64_t t = 0;                // Adam step count
    double *d_loss = nullptr, *h_loss = nullptr;
    std::vector<void *> bufs;
    // activations (bf16), dense, per level: encoder outputs of the two
    // convolutions, pooled input, decoder outputs
    uint16_t *ea[kLevels] = {}, *eb[kLevels] = {}, *pool[kLevels] = {}, *da[kLevels] = {}, *db[kLevels] = {};
    // output gradients (bf16): a layer reads one and writes the other
    uint16_t *dz[kLevels][2] = {};
    // gradients that meet another before they are rounded (FP32): skip
    // connections and pooled inputs
    float *g_skip[kLevels] = {}, *g_pool[kLevels] = {};

    int c(int l) const { return base << l; }
    int hl(int l) const { return H >> l; }
    int wl(int l) const { return W >> l; }
    int64_t pl(int l) const { return (int64_t)B * hl(l) * wl(l); }

    template <typename U>
    U *dalloc(int64_t count) {
        void *p = nullptr;
        LLGMI_HIP(hipMalloc(&p, sizeof(U) * (size_t)std::max<int64_t>(count, 1)));
        bufs.push_back(p);
        return (U *)p;
    }

    UNet(int B_, int H_, int W_, int cin_, int cout_, int base_, int wv_, int hv_, uint64_t seed)
        : B(B_), H(H_), W(W_), cin_real(cin_), cout_real(cout_), cout((cout_ + 15) / 16 * 16), base(base_),
          wv(wv_), hv(hv_) {
        try {
            LLGMI_HIP(hipStreamCreateWithFlags(&stream, hipStreamNonBlocking));
            // layers
            auto add = [&](int ci, int co, bool relu) {
                UNetConv cv;
                cv.cin = ci;
                cv.cout = co;
                cv.relu = relu;
                cv.w_off = nparam;
                nparam += (int64_t)9 * ci * co;
                cv.b_off = nparam;
                nparam += co;
                conv.push_back(cv);
            };
            for (int l = 0; l < kLevels; ++l) {
                add(l == 0 ? 16 : c(l - 1), c(l), true);
                add(c(l), c(l), true);
            }
            for (int l = kLevels - 2; l >= 0; --l) {
                add(c(l + 1) + c(l), c(l), true);
                add(c(l), c(l), true);
            }
            add(c(0), cout, false);
            d_p = dalloc<float>(nparam);
            d_g = dalloc<float>(nparam);
            d_m = dalloc<float>(nparam);
            d_v = dalloc<float>(nparam);
            int64_t nw = 0;
            for (auto &cv : conv) nw += 2 * (int64_t)9 * cv.cin * cv.cout;
            d_wbf = dalloc<uint16_t>(nw);
            int64_t o = 0;
            for (auto &cv : conv) {
                cv.wf = d_wbf + o;
                o += (int64_t)9 * cv.cin * cv.cout;
                cv.wb = d_wbf + o;
                o += (int64_t)9 * cv.cin * cv.cout;
            }
            int64_t npart = 0;
            for (size_t k = 0; k < conv.size(); ++k)
                npart = std::max(npart, wgrad_split(conv[k].cout, conv[k].cin, level_of((int)k)) *
                                            ((int64_t)9 * conv[k].cin * conv[k].cout + conv[k].cout));
            d_part = dalloc<float>(npart);
            d_loss = dalloc<double>(1);
            LLGMI_HIP(hipHostMalloc((void **)&h_loss, sizeof(double), hipHostMallocDefault));
            // activations and gradients
            for (int l = 0; l < kLevels; ++l) {
                const int64_t P = pl(l);
                ea[l] = dalloc<uint16_t>(P * c(l));
                eb[l] = dalloc<uint16_t>(P * c(l));
                if (l < kLevels - 1) {
                    da[l] = dalloc<uint16_t>(P * c(l));
                    db[l] = dalloc<uint16_t>(P * c(l));
                    g_skip[l] = dalloc<float>(P * c(l));
                }
                if (l > 0) {
                    pool[l] = dalloc<uint16_t>(P * c(l - 1));
                    g_pool[l] = dalloc<float>(P * c(l - 1));
                }
                for (auto &z : dz[l]) z = dalloc<uint16_t>(P * std::max(c(l), l == 0 ? cout : 0));
            }
            init(seed);
        } catch (...) {
            release();
            throw;
        }
    }
    ~UNet() { release(); }
    void release() {
        if (stream) (void)hipStreamSynchronize(stream);
        for (void *p : bufs) (void)hipFree(p);
        bufs.clear();
        if (h_loss) (void)hipHostFree(h_loss);
        h_loss = nullptr;
        if (stream) (void)hipStreamDestroy(stream);
        stream = nullptr;
    }

    // He-normal weights (std sqrt(2 / fan_in), fan_in over the real input
    // channels), the head scaled by 0.1; biases zero; padded channels zero.
    void init(uint64_t seed) {
        std::vector<float> h((size_t)nparam, 0.f);
        uint64_t s = seed ^ 0x9e3779b97f4a7c15ull;
        auto next = [&]() {   // xorshift64*
            s ^= s >> 12;
            s ^= s << 25;
            s ^= s >> 27;
            return (s * 0x2545f4914f6cdd1dull) >> 11;
        };
        auto uni = [&]() { return ((double)next() + 0.5) / 9007199254740992.0; };
        for (size_t k = 0; k < conv.size(); ++k) {
            const UNetConv &cv = conv[k];
            const bool first = k == 0, head = k + 1 == conv.size();
            const int fan = 9 * (first ? cin_real : cv.cin);
            const double sd = std::sqrt(2.0 / fan) * (head ? 0.1 : 1.0);
            for (int tap = 0; tap < 9; ++tap)
                for (int co = 0; co < cv.cout; ++co)
                    for (int ci = 0; ci < cv.cin; ++ci) {
                        const double u1 = uni(), u2 = uni();
                        const double gz = std::sqrt(-2.0 * std::log(u1)) * std::cos(6.283185307179586 * u2);
                        const bool live = (!first || ci < cin_real) && (!head || co < cout_real);
                        h[(size_t)(cv.w_off + ((int64_t)tap * cv.cout + co) * cv.cin + ci)] = live ? (float)(sd * gz) : 0.f;
                    }
        }
        set_params(h.data());
    }

    void set_params(const float *hp) {
        LLGMI_HIP(hipMemcpyAsync(d_p, hp, sizeof(float) * (size_t)nparam, hipMemcpyHostToDevice, stream));
        LLGMI_HIP(hipMemsetAsync(d_m, 0, sizeof(float) * (size_t)nparam, stream));
        LLGMI_HIP(hipMemsetAsync(d_v, 0, sizeof(float) * (size_t)nparam, stream));
        t = 0;
        cast_weights();
        LLGMI_HIP(hipStreamSynchronize(stream));
    }
    void cast_weights() {
        if (conv.size() != (size_t)kConvs) throw Error(LLGMI_ERR_INVALID, "internal: number of convolutions");
        CastLayers layers;
        for (int k = 0; k < kConvs; ++k) {
            const UNetConv &cv = conv[(size_t)k];
            layers.l[k] = CastLayer{cv.w_off, cv.cout, cv.cin, cv.wf, cv.wb};
        }
        hipLaunchKernelGGL(k_w_cast, dim3(128, kConvs), dim3(kNT), 0, stream, d_p, layers);
        LLGMI_LAUNCH_CHECK();
    }

    // ---- launch helpers with the shape checks the kernels rely on ----
    static ConvSrc dense(const uint16_t *x, int c) { return {nullptr, 0, x, c}; }
    static void check_src(const ConvSrc &s, int cin) {
        if (cin % 16 || s.lo_c + s.hi_c != cin || s.lo_c % kKC) throw Error(LLGMI_ERR_INVALID, "internal: convolution input");
    }

    template <int EPI, bool RELU>
    void conv3(ConvSrc src, int cin, const uint16_t *w, const float *bias, const ConvEpi &ep, int co, int l) {
        check_src(src, cin);
        // output channels per block: a divisor of the upsampled part too
        int nt = co % 32 == 0 ? 2 : co % 48 == 0 ? 3 : 1;
        if (EPI == EPI_CAT && ep.up_c % (16 * nt)) nt = 1;
        if (co % (16 * nt) || (EPI == EPI_CAT && ep.up_c % (16 * nt)))
            throw Error(LLGMI_ERR_INVALID, "internal: convolution shape");
        if ((ep.pool || EPI == EPI_CAT) && (hl(l) % 2 || wl(l) % 2)) throw Error(LLGMI_ERR_INVALID, "internal: odd plane");
        // Pixel tile: the largest that gives two blocks to every CU twice over;
        // 16 x 32 reads least per product, but on narrow planes its padding
        // (columns past the image) costs more than that.  LLGMI_UNET_TILE=8x16 (or
        // 0), 16x16 or 16x32 takes that tile everywhere (16x32 where it is built).
        auto tiles = [&](int th, int tw) {
            return (int64_t)B * ((hl(l) + th - 1) / th) * ((wl(l) + 16 * tw - 1) / (16 * tw));
        };
        const int64_t groups = co / (16 * nt);
        bool wide = nt < 3 && tiles(16, 2) * groups >= 1024 && 10 * 2 * tiles(16, 2) <= 11 * tiles(16, 1);
        bool tall = tiles(16, 1) * groups >= 512;
        if (const char *e = std::getenv("LLGMI_UNET_TILE")) {
            const std::string v(e);
            const bool w32 = v == "16x32";
            if (w32 || v == "16x16" || v == "8x16" || v[0] == '0') {
                wide = w32 && nt < 3;
                tall = w32 || v == "16x16";
            }
        }
        auto go = [&](auto ntc) {
            constexpr int NT = decltype(ntc)::value;
            if (wide) {
                if constexpr (NT < 3) launch_conv<16, 2, NT, EPI, RELU>(src, cin, w, bias, ep, co, l);
            } else if (tall) launch_conv<16, 1, NT, EPI, RELU>(src, cin, w, bias, ep, co, l);
            else launch_conv<8, 1, NT, EPI, RELU>(src, cin, w, bias, ep, co, l);
        };
        if (nt == 3) go(std::integral_constant<int, 3>{});
        else if (nt == 2) go(std::integral_constant<int, 2>{});
        else go(std::integral_constant<int, 1>{});
    }
    template <int TH, int TW, int NT, int EPI, bool RELU>
    void launch_conv(ConvSrc src, int cin, const uint16_t *w, const float *bias, const ConvEpi &ep, int co, int l) {
        constexpr size_t lds = ConvShape<TH, TW, NT>::LDS;
        auto kern = k_conv3x3<TH, TW, NT, EPI, RELU>;
        {
            // the LDS attribute is set once per kernel and device
            static std::mutex mu;
            static std::set<int> done;
            int dev = 0;
            LLGMI_HIP(hipGetDevice(&dev));
            std::lock_guard<std::mutex> lock(mu);
            if (!done.count(dev)) {
                LLGMI_HIP(hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
                done.insert(dev);
            }
        }
        const int ntile = ((wl(l) + 16 * TW - 1) / (16 * TW)) * ((hl(l) + TH - 1) / TH) * B, groups = co / (16 * NT);
        // one-chunk layers run several tiles per block (weights stay in LDS): as
        // many as leave one round of resident blocks, the same number each
        const int64_t slots = 256 * conv_blocks_per_cu<TW, NT>();
        const int per = cin <= kKC ? (int)(((int64_t)ntile * groups + slots - 1) / slots) : 1;
        const int nb = (ntile + per - 1) / per;
        hipLaunchKernelGGL(kern, dim3((unsigned)nb, (unsigned)groups), dim3(256), lds, stream, src, cin, w, bias, ep, co,
                           B, hl(l), wl(l));
        LLGMI_LAUNCH_CHECK();
    }
    // forward of a hidden layer: bf16 relu(conv + bias) to y, and its average pool
    void act(ConvSrc src, const UNetConv &cv, uint16_t *y, int l, uint16_t *pooled = nullptr) {
        ConvEpi ep;
        ep.y = y;
        ep.pool = pooled;
        conv3<EPI_ACT, true>(src, cv.cin, cv.wf, d_p + cv.b_off, ep, cv.cout, l);
    }
    // data gradient of cv from dz, masked by the activation it flows into
    void dgrad(const uint16_t *dzp, const UNetConv &cv, const uint16_t *mask, uint16_t *y, int l) {
        ConvEpi ep;
        ep.y = y;
        ep.mask = mask;
        conv3<EPI_MASK, false>(dense(dzp, cv.cout), cv.cout, cv.wb, nullptr, ep, cv.cin, l);
    }
    void wgrad(const uint16_t *dzp, ConvSrc src, const UNetConv &cv, int l) {
        const int co = cv.cout, ci = cv.cin;
        check_src(src, ci);
        if (co % 16) throw Error(LLGMI_ERR_INVALID, "internal: weight-gradient shape");
        const int mt = wgrad_mt(co), nt = wgrad_nt(co, ci);
        const dim3 grid((unsigned)wgrad_split(co, ci, l), (unsigned)((co / (16 * mt)) * (ci / (16 * nt))));
        auto go = [&](auto kern) {
            hipLaunchKernelGGL(kern, grid, dim3(256), 0, stream, dzp, co, src, ci, d_part, B, hl(l), wl(l));
        };
        if (mt == 3) go(k_conv3x3_wgrad<3, 1>);
        else if (mt == 2) nt == 2 ? go(k_conv3x3_wgrad<2, 2>) : go(k_conv3x3_wgrad<2, 1>);
        else nt == 2 ? go(k_conv3x3_wgrad<1, 2>) : go(k_conv3x3_wgrad<1, 1>);
        // a layer's weights and bias are consecutive in the parameter vector
        const int64_t n = (int64_t)9 * co * ci + co;
        hipLaunchKernelGGL(k_part_sum, dim3((unsigned)((n + 63) / 64)), dim3(256), 0, stream, d_part, (int)grid.x, n,
                           d_g + cv.w_off);
        LLGMI_LAUNCH_CHECK();
    }
    // channel tiles of the weight gradient (48 output channels in one tile of
    // three, then with one input tile: three by two spill) and the pixel runs a layer is split into: two blocks per CU in all,
    // no more than there are pixel tiles, a multiple of the eight XCDs so that
    // the channel tiles of one run share an L2
    static int wgrad_mt(int co) { return co % 32 == 0 ? 2 : co % 48 == 0 ? 3 : 1; }
    static int wgrad_nt(int co, int ci) { return wgrad_mt(co) < 3 && ci % 32 == 0 ? 2 : 1; }
    int wgrad_split(int co, int ci, int l) const {
        const int64_t tiles = (int64_t)B * ((hl(l) + kWgT - 1) / kWgT) * ((wl(l) + kWgT - 1) / kWgT);
        int64_t s = std::max<int64_t>(1, 512 / ((co / (16 * wgrad_mt(co))) * (ci / (16 * wgrad_nt(co, ci)))));
        if (s > 8) s -= s % 8;
        return (int)std::min(s, tiles);
    }

    // conv index: enc l -> 2l, 2l+1; dec l (2..0) -> 8 + 2(2-l), +1; head -> 14
    const UNetConv &enc(int l, int k) const { return conv[(size_t)(2 * l + k)]; }
    const UNetConv &dec(int l, int k) const { return conv[(size_t)(2 * kLevels + 2 * (kLevels - 2 - l) + k)]; }
    const UNetConv &head() const { return conv.back(); }
    static int level_of(int k) { return k < 2 * kLevels ? k / 2 : k == kConvs - 1 ? 0 : kLevels - 2 - (k - 2 * kLevels) / 2; }

    // decoder l's input: the upsampled level below and enc_l's output
    ConvSrc cat(int l) const { return {l == kLevels - 2 ? eb[l + 1] : db[l + 1], c(l + 1), eb[l], c(l)}; }

    // every layer but the head
    void trunk(const uint16_t *x) {
        for (int l = 0; l < kLevels; ++l) {
            act(l == 0 ? dense(x, 16) : dense(pool[l], c(l - 1)), enc(l, 0), ea[l], l);
            act(dense(ea[l], c(l)), enc(l, 1), eb[l], l, l + 1 < kLevels ? pool[l + 1] : nullptr);
        }
        for (int l = kLevels - 2; l >= 0; --l) {
            act(cat(l), dec(l, 0), da[l], l);
            act(dense(da[l], c(l)), dec(l, 1), db[l], l);
        }
    }
    void forward(const uint16_t *x, float *y) {
        trunk(x);
        ConvEpi ep;
        ep.yf = y;
        conv3<EPI_F32, false>(dense(db[0], c(0)), c(0), head().wf, d_p + head().b_off, ep, cout, 0);
    }

    // gradient of the loss w.r.t. every parameter into d_g (overwritten)
    double loss_grad(const uint16_t *x, const uint16_t *tgt) {
        LLGMI_HIP(hipMemsetAsync(d_loss, 0, sizeof(double), stream));
        trunk(x);
        {
            // head with the loss and its gradient
            ConvEpi ep;
            ep.y = dz[0][0];
            ep.tgt = tgt;
            ep.cv = cout_real;
            ep.wv = wv;
            ep.hv = hv;
            ep.inv_count = 1.0 / ((double)B * wv * hv * cout_real);
            ep.loss = d_loss;
            conv3<EPI_MSE, false>(dense(db[0], c(0)), c(0), head().wf, d_p + head().b_off, ep, cout, 0);
        }
        LLGMI_HIP(hipMemcpyAsync(h_loss, d_loss, sizeof(double), hipMemcpyDeviceToHost, stream));
        wgrad(dz[0][0], dense(db[0], c(0)), head(), 0);
        dgrad(dz[0][0], head(), db[0], dz[0][1], 0);
        // decoders, top level first; dz[l][1] holds the gradient of dec_l's output
        for (int l = 0; l <= kLevels - 2; ++l) {
            wgrad(dz[l][1], dense(da[l], c(l)), dec(l, 1), l);
            dgrad(dz[l][1], dec(l, 1), da[l], dz[l][0], l);
            wgrad(dz[l][0], cat(l), dec(l, 0), l);
            // up part: masked gradient of the level below's output; skip part: to be joined by the pool's
            ConvEpi ep;
            ep.y = dz[l + 1][1];
            ep.mask = cat(l).lo;
            ep.up_c = c(l + 1);
            ep.yf = g_skip[l];
            conv3<EPI_CAT, false>(dense(dz[l][0], c(l)), c(l), dec(l, 0).wb, nullptr, ep, dec(l, 0).cin, l);
        }
        // encoders, bottom level first; dz[l][1] holds the gradient of enc_l's output
        for (int l = kLevels - 1; l >= 0; --l) {
            if (l < kLevels - 1) {
                hipLaunchKernelGGL(k_skip_pool_relu, dim3(grid_of(pl(l) * c(l) / 8)), dim3(kNT), 0, stream, g_skip[l],
                                   g_pool[l + 1], eb[l], c(l), dz[l][1], B, hl(l), wl(l));
                LLGMI_LAUNCH_CHECK();
            }
            wgrad(dz[l][1], dense(ea[l], c(l)), enc(l, 1), l);
            dgrad(dz[l][1], enc(l, 1), ea[l], dz[l][0], l);
            if (l == 0) {
                wgrad(dz[0][0], dense(x, 16), enc(0, 0), 0);
            } else {
                wgrad(dz[l][0], dense(pool[l], c(l - 1)), enc(l, 0), l);
                ConvEpi ep;
                ep.yf = g_pool[l];
                conv3<EPI_F32, false>(dense(dz[l][0], c(l)), c(l), enc(l, 0).wb, nullptr, ep, c(l - 1), l);
            }
        }
        LLGMI_HIP(hipStreamSynchronize(stream));
        return *h_loss;
    }

    void adam(double lr) {
        ++t;
        const float b1 = 0.9f, b2 = 0.999f;
        const float bc1 = 1.f - std::pow(b1, (float)t), bc2 = 1.f - std::pow(b2, (float)t);
        hipLaunchKernelGGL(k_adam, dim3(grid_of(nparam)), dim3(kNT), 0, stream, d_p, d_g, d_m, d_v, nparam,
                           (float)lr, b1, b2, 1e-8f, bc1, bc2);
        cast_weights();
        LLGMI_LAUNCH_CHECK();
    }
};

}  // namespace llgmi

// ---------------------------------------------------------------------------
// C ABI
// ---------------------------------------------------------------------------
using llgmi::Error;
using llgmi::UNet;

struct llgmi_ws {
    std::unique_ptr<UNet> net;
    int device = 0;
};

namespace {
int ws_fail(int code, const std::string &m) { return llgmi::set_last_error(code, m); }

void need(const void *p, int64_t bytes, const char *what) {
    const std::string e = llgmi::check_device_range(p, (size_t)bytes, what);
    if (!e.empty()) throw Error(LLGMI_ERR_INVALID, e);
}
int64_t x_bytes(const UNet &u) { return u.pl(0) * 16 * 2; }
int64_t t_bytes(const UNet &u) { return u.pl(0) * u.cout * 2; }
int64_t y_bytes(const UNet &u) { return u.pl(0) * u.cout * 4; }

template <typename F>
int ws_guard(llgmi_ws *ws, F &&f) {
    if (!ws || !ws->net) return ws_fail(LLGMI_ERR_INVALID, "warm-start network is NULL");
    try {
        LLGMI_HIP(hipSetDevice(ws->device));
        f(*ws->net);
        return LLGMI_OK;
    } catch (const Error &e) {
        return ws_fail(e.code, e.what());
    } catch (const std::bad_alloc &) {
        return ws_fail(LLGMI_ERR_ALLOC, "host allocation failed");
    } catch (const std::exception &e) {
        return ws_fail(LLGMI_ERR_INVALID, e.what());
    }
}
}  // namespace

extern "C" {

int llgmi_ws_create(const llgmi_ws_shape *shape, uint64_t seed, int device, llgmi_ws **out) {
    if (!shape || !out) return ws_fail(LLGMI_ERR_INVALID, "NULL argument");
    *out = nullptr;
    const llgmi_ws_shape &s = *shape;
    const int64_t div = (int64_t)1 << (llgmi::kLevels - 1);
    if (s.batch < 1 || s.height < div || s.width < div || s.height % div || s.width % div)
        return ws_fail(LLGMI_ERR_INVALID, "height and width must be positive multiples of 8, batch >= 1");
    if (s.in_channels < 1 || s.in_channels > 16) return ws_fail(LLGMI_ERR_INVALID, "in_channels must be 1..16");
    if (s.out_channels < 1 || s.out_channels > 256) return ws_fail(LLGMI_ERR_INVALID, "out_channels must be 1..256");
    if (s.base_channels < 16 || s.base_channels % 16 || s.base_channels > 32)
        return ws_fail(LLGMI_ERR_INVALID, "base_channels must be 16 or 32");
    if (s.batch * s.height * s.width > ((int64_t)1 << 28)) return ws_fail(LLGMI_ERR_INVALID, "batch too large");
    if (s.valid_width < 1 || s.valid_height < 1) return ws_fail(LLGMI_ERR_INVALID, "valid region is empty");
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || device < 0 || device >= ndev)
        return ws_fail(LLGMI_ERR_INVALID, "device index out of range");
    std::unique_ptr<llgmi_ws> ws(new (std::nothrow) llgmi_ws());
    if (!ws) return ws_fail(LLGMI_ERR_ALLOC, "host allocation failed");
    ws->device = device;
    try {
        LLGMI_HIP(hipSetDevice(device));
        // a valid region beyond the plane is the whole plane
        ws->net.reset(new UNet((int)s.batch, (int)s.height, (int)s.width, s.in_channels, s.out_channels,
                               s.base_channels, (int)std::min(s.valid_width, s.width),
                               (int)std::min(s.valid_height, s.height), seed));
    } catch (const Error &e) {
        return ws_fail(e.code, e.what());
    } catch (const std::bad_alloc &) {
        return ws_fail(LLGMI_ERR_ALLOC, "host allocation failed");
    }
    *out = ws.release();
    return LLGMI_OK;
}

int llgmi_ws_destroy(llgmi_ws *ws) {
    if (!ws) return LLGMI_OK;
    (void)hipSetDevice(ws->device);
    ws->net.reset();
    delete ws;
    return LLGMI_OK;
}

int llgmi_ws_param_count(llgmi_ws *ws, int64_t *n) {
    if (!n) return ws_fail(LLGMI_ERR_INVALID, "NULL argument");
    return ws_guard(ws, [&](UNet &u) { *n = u.nparam; });
}

int llgmi_ws_get_params(llgmi_ws *ws, float *host) {
    if (!host) return ws_fail(LLGMI_ERR_INVALID, "NULL argument");
    return ws_guard(ws, [&](UNet &u) {
        LLGMI_HIP(hipMemcpyAsync(host, u.d_p, sizeof(float) * (size_t)u.nparam, hipMemcpyDeviceToHost, u.stream));
        LLGMI_HIP(hipStreamSynchronize(u.stream));
    });
}

int llgmi_ws_set_params(llgmi_ws *ws, const float *host) {
    if (!host) return ws_fail(LLGMI_ERR_INVALID, "NULL argument");
    return ws_guard(ws, [&](UNet &u) { u.set_params(host); });
}

int llgmi_ws_get_grads(llgmi_ws *ws, float *host) {
    if (!host) return ws_fail(LLGMI_ERR_INVALID, "NULL argument");
    return ws_guard(ws, [&](UNet &u) {
        LLGMI_HIP(hipMemcpyAsync(host, u.d_g, sizeof(float) * (size_t)u.nparam, hipMemcpyDeviceToHost, u.stream));
        LLGMI_HIP(hipStreamSynchronize(u.stream));
    });
}

int llgmi_ws_forward(llgmi_ws *ws, const uint16_t *x_dev, float *y_dev) {
    if (!x_dev || !y_dev) return ws_fail(LLGMI_ERR_INVALID, "NULL buffer");
    return ws_guard(ws, [&](UNet &u) {
        need(x_dev, x_bytes(u), "x");
        need(y_dev, y_bytes(u), "y");
        u.forward(x_dev, y_dev);
        LLGMI_HIP(hipStreamSynchronize(u.stream));
    });
}

int llgmi_ws_loss_grad(llgmi_ws *ws, const uint16_t *x_dev, const uint16_t *t_dev, double *loss) {
    if (!x_dev || !t_dev || !loss) return ws_fail(LLGMI_ERR_INVALID, "NULL argument");
    return ws_guard(ws, [&](UNet &u) {
        need(x_dev, x_bytes(u), "x");
        need(t_dev, t_bytes(u), "t");
        *loss = u.loss_grad(x_dev, t_dev);
    });
}

int llgmi_ws_adam_step(llgmi_ws *ws, double lr) {
    if (!(lr > 0.0)) return ws_fail(LLGMI_ERR_INVALID, "learning rate must be positive");
    return ws_guard(ws, [&](UNet &u) {
        u.adam(lr);
        LLGMI_HIP(hipStreamSynchronize(u.stream));
    });
}

int llgmi_ws_train_step(llgmi_ws *ws, const uint16_t *x_dev, const uint16_t *t_dev, double lr, double *loss) {
    if (!x_dev || !t_dev || !loss) return ws_fail(LLGMI_ERR_INVALID, "NULL argument");
    if (!(lr > 0.0)) return ws_fail(LLGMI_ERR_INVALID, "learning rate must be positive");
    return ws_guard(ws, [&](UNet &u) {
        need(x_dev, x_bytes(u), "x");
        need(t_dev, t_bytes(u), "t");
        *loss = u.loss_grad(x_dev, t_dev);
        u.adam(lr);
        LLGMI_HIP(hipStreamSynchronize(u.stream));
    });
}

int llgmi_ws_pack_input(llgmi_ws *ws, int64_t sample, const void *m_dev, int m_is_f32, int64_t nx, int64_t ny,
                        int64_t offx, int64_t offy, uint16_t *x_dev) {
    if (!m_dev || !x_dev) return ws_fail(LLGMI_ERR_INVALID, "NULL buffer");
    return ws_guard(ws, [&](UNet &u) {
        if (sample < 0 || sample >= u.B) throw Error(LLGMI_ERR_INVALID, "sample index out of range");
        if (nx < 1 || ny < 1 || offx < 0 || offy < 0 || offx + nx > u.W || offy + ny > u.H)
            throw Error(LLGMI_ERR_INVALID, "film does not fit the network's plane");
        need(m_dev, 3 * nx * ny * (m_is_f32 ? 4 : 8), "m");
        need(x_dev, x_bytes(u), "x");
        uint16_t *dst = x_dev + sample * (int64_t)u.H * u.W * 16;
        const int64_t n = (int64_t)u.H * u.W;
        if (m_is_f32)
            hipLaunchKernelGGL(llgmi::k_pack_input<float>, dim3(llgmi::grid_of(n)), dim3(256), 0, u.stream,
                               (const float *)m_dev, (int)nx, (int)ny, (int)offx, (int)offy, dst, u.H, u.W);
        else
            hipLaunchKernelGGL(llgmi::k_pack_input<double>, dim3(llgmi::grid_of(n)), dim3(256), 0, u.stream,
                               (const double *)m_dev, (int)nx, (int)ny, (int)offx, (int)offy, dst, u.H, u.W);
        LLGMI_LAUNCH_CHECK();
        LLGMI_HIP(hipStreamSynchronize(u.stream));
    });
}

int llgmi_ws_pack_phi(llgmi_ws *ws, int64_t sample, const double *phi_dev, int64_t px, int64_t py, int64_t pz,
                      double scale, uint16_t *t_dev) {
    if (!phi_dev || !t_dev) return ws_fail(LLGMI_ERR_INVALID, "NULL buffer");
    if (!(scale > 0.0)) return ws_fail(LLGMI_ERR_INVALID, "scale must be positive");
    return ws_guard(ws, [&](UNet &u) {
        if (sample < 0 || sample >= u.B) throw Error(LLGMI_ERR_INVALID, "sample index out of range");
        if (px < 1 || py < 1 || pz < 1 || px > u.W || py > u.H || pz > u.cout_real)
            throw Error(LLGMI_ERR_INVALID, "box does not fit the network's plane and channels");
        need(phi_dev, px * py * pz * 8, "phi");
        need(t_dev, t_bytes(u), "t");
        uint16_t *dst = t_dev + sample * (int64_t)u.H * u.W * u.cout;
        const int64_t n = (int64_t)u.H * u.W * u.cout;
        hipLaunchKernelGGL(llgmi::k_pack_phi, dim3(llgmi::grid_of(n)), dim3(256), 0, u.stream, phi_dev, (int)px,
                           (int)py, (int)pz, 1.0 / scale, dst, u.cout, u.H, u.W);
        LLGMI_LAUNCH_CHECK();
        LLGMI_HIP(hipStreamSynchronize(u.stream));
    });
}

int llgmi_ws_unpack_phi(llgmi_ws *ws, int64_t sample, const float *y_dev, int64_t px, int64_t py, int64_t pz,
                        double scale, int accumulate, double *phi_dev) {
    if (!phi_dev || !y_dev) return ws_fail(LLGMI_ERR_INVALID, "NULL buffer");
    return ws_guard(ws, [&](UNet &u) {
        if (sample < 0 || sample >= u.B) throw Error(LLGMI_ERR_INVALID, "sample index out of range");
        if (px < 1 || py < 1 || pz < 1 || px > u.W || py > u.H || pz > u.cout_real)
            throw Error(LLGMI_ERR_INVALID, "box does not fit the network's plane and channels");
        need(phi_dev, px * py * pz * 8, "phi");
        need(y_dev, y_bytes(u), "y");
        const float *src = y_dev + sample * (int64_t)u.H * u.W * u.cout;
        const int64_t n = px * py * pz;
        hipLaunchKernelGGL(llgmi::k_unpack_phi, dim3(llgmi::grid_of(n)), dim3(256), 0, u.stream, src, u.cout, u.H,
                           u.W, scale, accumulate, phi_dev, (int)px, (int)py, (int)pz);
        LLGMI_LAUNCH_CHECK();
        LLGMI_HIP(hipStreamSynchronize(u.stream));
    });
}

}  // extern "C"
