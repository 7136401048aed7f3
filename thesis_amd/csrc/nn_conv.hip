// 3x3 (and 1x1) convolutions of the warm-start network as implicit GEMMs on
// bf16 MFMA: the im2col matrix is never stored.
//
// A workgroup of four waves owns TY image rows x 32 pixels of one image.  It
// loads their inputs with a one-pixel frame once, rounds them to bf16 into LDS
// (pixel-major, all input channels) and walks the taps: the A operand of a tap
// is the same LDS patch read one pixel further, the B operand the tap's weights,
// read from L2 (each wave's own columns; 18-295 KB a layer).  One LDS read of
// a pixel serves nine taps, where im2col wrote and read it nine times.
//
// Prediction of 8 channels of 512 x 128: 3.11 -> 0.63 ms against im2col (55 % of
// the time) + GEMM + upsampling and skip-sum passes; a training step on 16:
// 21.4 -> 3.4 ms.  What bounds it now: the FP32 activations' traffic at full
// resolution (32 channels); at the coarse levels the latency of staging and
// weights, one or two workgroups a CU (128 channels: 34 us of which 8 are MFMA).
// Weights staged in LDS for the four waves cost more in barriers and in
// workgroups a CU than they saved (43 us), loads six steps ahead gave nothing.
//
// The sums run in the order of the im2col GEMM (tap, then channel, 16 at a time
// in v_mfma_f32_32x32x16_bf16), so outputs are the same bits.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>

#include "lbm_nn.h"

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4), aligned(4)));   // rows may start at any float
typedef uint16_t u16;

constexpr int TX = 32;   // pixels of a tile row: the 32 rows of an MFMA operand

// Rounded to nearest even by v_cvt_pk_bf16_f32: half an instruction a value, where
// the same rounding in integer arithmetic took about eight and the staging of a
// tile as long as its MFMA.
__device__ inline uint2 f2bf4(f32x4 v) {
    typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
    return __builtin_bit_cast(uint2, bf16x4{(__bf16)v[0], (__bf16)v[1], (__bf16)v[2], (__bf16)v[3]});
}

// Input of a convolution: x itself, x at half the resolution (each pixel read by
// the 2 x 2 it covers), or x + skip.
enum { IN_X = 0, IN_UP = 1, IN_ADD = 2 };
struct Img {
    const float* x;
    const float* skip;
    int H, W, C;
};
template <int MODE>
__device__ inline f32x4 fetch(const Img& s, int b, int y, int x, int c) {
    if (MODE == IN_UP)
        return *(const f32x4*)(s.x + (((size_t)b * (s.H >> 1) + (y >> 1)) * (s.W >> 1) + (x >> 1)) * s.C + c);
    const size_t i = (((size_t)b * s.H + y) * s.W + x) * s.C + c;
    f32x4 v = *(const f32x4*)(s.x + i);
    if (MODE == IN_ADD) {
        const f32x4 w = *(const f32x4*)(s.skip + i);
        v = f32x4{v[0] + w[0], v[1] + w[1], v[2] + w[2], v[3] + w[3]};
    }
    return v;
}

// The staging loops below load from the nearest pixel inside the image and zero
// what lies outside after the load, U loads of a thread at a time: a load under a
// branch would be waited for before the next is issued (weight gradients of a
// training step 1.55 -> 0.99 ms, forward convolutions of a prediction 0.64 -> 0.57).
__device__ inline int clampi(int a, int n) { return a < 0 ? 0 : (a >= n ? n - 1 : a); }

// Channels c0 .. c0+KC-1 of the ROWS x COLS pixels at (y0, x0) as bf16 in LDS,
// zero outside the image; pitch P.
template <int KC, int P, int ROWS, int COLS, int MODE, int U>
__device__ inline void stage(const Img& s, int b, int y0, int x0, int c0, u16* t) {
    constexpr int V = KC / 4, N = ROWS * COLS * V, NV = (N + 255) / 256;
    for (int i0 = 0; i0 < NV; i0 += U) {
        f32x4 e[U];
        bool in[U];
#pragma unroll
        for (int i = 0; i < U; ++i) {
            const int v0 = threadIdx.x + 256 * (i0 + i), v = v0 < N ? v0 : N - 1;
            const int px = v / V, c = (v - px * V) * 4, r = px / COLS;
            const int y = y0 + r, x = x0 + px - r * COLS;
            in[i] = y >= 0 && y < s.H && x >= 0 && x < s.W;
            e[i] = fetch<MODE>(s, b, clampi(y, s.H), clampi(x, s.W), c0 + c);
        }
#pragma unroll
        for (int i = 0; i < U; ++i) {
            const int v = threadIdx.x + 256 * (i0 + i), px = v / V, c = (v - px * V) * 4;
            const uint2 q = f2bf4(e[i]);
            if (v < N) *(uint2*)(t + px * P + c) = in[i] ? q : make_uint2(0u, 0u);
        }
    }
}
// The same of a bf16 image (8 channels a load).
template <int KC, int P, int ROWS, int COLS, int U>
__device__ inline void stage_bf(const u16* __restrict__ z, int H, int W, int C, int b, int y0, int x0, int c0, u16* t) {
    constexpr int V = KC / 8, N = ROWS * COLS * V, NV = (N + 255) / 256;
    for (int i0 = 0; i0 < NV; i0 += U) {
        uint4 e[U];
        bool in[U];
#pragma unroll
        for (int i = 0; i < U; ++i) {
            const int v0 = threadIdx.x + 256 * (i0 + i), v = v0 < N ? v0 : N - 1;
            const int px = v / V, c = (v - px * V) * 8, r = px / COLS;
            const int y = y0 + r, x = x0 + px - r * COLS;
            in[i] = y >= 0 && y < H && x >= 0 && x < W;
            e[i] = *(const uint4*)(z + (((size_t)b * H + clampi(y, H)) * W + clampi(x, W)) * C + c0 + c);
        }
#pragma unroll
        for (int i = 0; i < U; ++i) {
            const int v = threadIdx.x + 256 * (i0 + i), px = v / V, c = (v - px * V) * 8;
            if (v < N) *(uint4*)(t + px * P + c) = in[i] ? e[i] : make_uint4(0u, 0u, 0u, 0u);
        }
    }
}
// Four input channels: the nine taps of a pixel side by side (36 of KC columns,
// the rest zero), so that the patch is a matrix row per pixel.
template <int KC, int P, int ROWS, int U>
__device__ inline void stage_taps(const Img& s, int b, int y0, int x0, u16* t) {
    constexpr int V = KC / 4, N = ROWS * TX * V, NV = (N + 255) / 256;
    for (int i0 = 0; i0 < NV; i0 += U) {
        f32x4 e[U];
        bool in[U];
#pragma unroll
        for (int i = 0; i < U; ++i) {
            const int v0 = threadIdx.x + 256 * (i0 + i), v = v0 < N ? v0 : N - 1;
            const int px = v / V, tap = v - px * V, r = px / TX, ky = tap / 3;
            const int y = y0 + r + ky - 1, x = x0 + px - r * TX + (tap - 3 * ky) - 1;
            in[i] = tap < 9 && y >= 0 && y < s.H && x >= 0 && x < s.W;
            e[i] = fetch<IN_X>(s, b, clampi(y, s.H), clampi(x, s.W), 0);
        }
#pragma unroll
        for (int i = 0; i < U; ++i) {
            const int v = threadIdx.x + 256 * (i0 + i), px = v / V, tap = v - px * V;
            const uint2 q = f2bf4(e[i]);
            if (v < N) *(uint2*)(t + px * P + tap * 4) = in[i] ? q : make_uint2(0u, 0u);
        }
    }
}

struct Tile {
    int b, y0, x0;
};
// tile index -> image and corner; tx, ty tiles per row and column
__device__ inline Tile tile_of(uint32_t t, uint32_t tx, uint32_t ty, int TY) {
    const uint32_t q = t / tx, b = q / ty;
    return Tile{(int)b, (int)(q - b * ty) * TY, (int)(t - q * tx) * TX};
}

// Forward convolution (KIND 0: 3x3; 1: 3x3 of four channels, KC = 48 of the 64
// weight columns; 2: 1x1).  Waves WM x WN, each TM image rows x TN blocks of 32
// output channels.
template <int KIND, int KC, int TY, int WM, int WN, int TM, int TN, int MODE>
__global__ __launch_bounds__(256) void k_conv(Img s, const u16* __restrict__ w, int kp, const float* __restrict__ bias,
                                              int relu, int N, uint32_t tx, uint32_t ty, float* __restrict__ y) {
    static_assert(WM * WN == 4 && WM * TM == TY, "four waves over the tile's rows");
    constexpr int HALO = KIND == 0 ? 1 : 0, COLS = TX + 2 * HALO, ROWS = TY + 2 * HALO, P = KC + 8;
    constexpr int TAPS = KIND == 0 ? 9 : 1;
    __shared__ __align__(16) u16 t[ROWS * COLS * P];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, wm = wave / WN, wn = wave % WN;
    const Tile tl = tile_of(blockIdx.x, tx, ty, TY);
    if (KIND == 1) stage_taps<KC, P, ROWS, 6>(s, tl.b, tl.y0, tl.x0, t);
    else stage<KC, P, ROWS, COLS, MODE, MODE == IN_ADD ? 4 : 8>(s, tl.b, tl.y0 - HALO, tl.x0 - HALO, 0, t);
    f32x16 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;
    const int ko = 8 * (lane >> 5), px = lane & 31;
    const u16* wp[TN];
    bool col[TN];
#pragma unroll
    for (int j = 0; j < TN; ++j) {
        const int n = (wn * TN + j) * 32 + px;
        col[j] = n < N;
        wp[j] = w + (size_t)(col[j] ? n : 0) * kp + ko;
    }
    __syncthreads();
#pragma unroll 3
    for (int tap = 0; tap < TAPS; ++tap) {
        const int ky = tap / 3, kx = tap - 3 * ky;
        const u16* ap = t + ((wm * TM + ky) * COLS + px + kx) * P + ko;
#pragma unroll
        for (int k = 0; k < KC; k += 16) {
            bf16x8 a[TM], b[TN];
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                uint4 v = *(const uint4*)(wp[j] + tap * KC + k);
                if (KIND == 2 && !col[j]) v = make_uint4(0u, 0u, 0u, 0u);   // N = 3: columns beyond are zero
                b[j] = __builtin_bit_cast(bf16x8, v);
            }
#pragma unroll
            for (int i = 0; i < TM; ++i) a[i] = *(const bf16x8*)(ap + i * COLS * P + k);
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[i], b[j], acc[i][j], 0, 0, 0);
        }
    }
#pragma unroll
    for (int i = 0; i < TM; ++i) {
        const int yy = tl.y0 + wm * TM + i;
        if (yy >= s.H) continue;
        float* row = y + ((size_t)tl.b * s.H + yy) * s.W * N;
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            const int n = (wn * TN + j) * 32 + px;
            if (n >= N) continue;
            const float bn = bias[n];
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int x = tl.x0 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
                if (x >= s.W) continue;
                float v = acc[i][j][r] + bn;
                if (relu) v = fmaxf(v, 0.f);
                row[(size_t)x * N + n] = v;
            }
        }
    }
}

// Input gradient of a 3x3 convolution: dx[p][c] = sum over taps of the product
// of dz at the output pixel that read p with the tap's weights wt[tap][c][n].
// Each tap's product is summed from zero and the taps added in order, as the
// stored products of every tap and col2im did.  KC: output channels of the
// convolution (the reduction), N: its input channels.
template <int KC, int TY, int WM, int WN, int TM, int TN>
__global__ __launch_bounds__(256) void k_conv_dx(const u16* __restrict__ dz, int H, int W, const u16* __restrict__ wt,
                                                 int N, uint32_t tx, uint32_t ty, float* __restrict__ dx) {
    static_assert(WM * WN == 4 && WM * TM == TY, "four waves over the tile's rows");
    constexpr int COLS = TX + 2, ROWS = TY + 2, P = KC + 8;
    __shared__ __align__(16) u16 t[ROWS * COLS * P];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, wm = wave / WN, wn = wave % WN;
    const Tile tl = tile_of(blockIdx.x, tx, ty, TY);
    stage_bf<KC, P, ROWS, COLS, 6>(dz, H, W, KC, tl.b, tl.y0 - 1, tl.x0 - 1, 0, t);
    f32x16 tot[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) tot[i][j][r] = 0.f;
    const int ko = 8 * (lane >> 5), px = lane & 31;
    const u16* wp = wt + (size_t)(wn * TN * 32 + px) * KC + ko;
    __syncthreads();
#pragma unroll 1
    for (int tap = 0; tap < 9; ++tap) {
        const int ky = tap / 3, kx = tap - 3 * ky;
        const u16* ap = t + ((wm * TM + 2 - ky) * COLS + px + 2 - kx) * P + ko;
        const u16* bp = wp + (size_t)tap * N * KC;
        f32x16 acc[TM][TN];
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j)
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;
#pragma unroll
        for (int k = 0; k < KC; k += 16) {
            bf16x8 a[TM], b[TN];
#pragma unroll
            for (int j = 0; j < TN; ++j) b[j] = *(const bf16x8*)(bp + j * 32 * KC + k);
#pragma unroll
            for (int i = 0; i < TM; ++i) a[i] = *(const bf16x8*)(ap + i * COLS * P + k);
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[i], b[j], acc[i][j], 0, 0, 0);
        }
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j)
#pragma unroll
                for (int r = 0; r < 16; ++r) tot[i][j][r] += acc[i][j][r];
    }
#pragma unroll
    for (int i = 0; i < TM; ++i) {
        const int yy = tl.y0 + wm * TM + i;
        if (yy >= H) continue;
        float* row = dx + ((size_t)tl.b * H + yy) * W * N;
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            const int n = (wn * TN + j) * 32 + px;
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int x = tl.x0 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
                if (x < W) row[(size_t)x * N + n] = tot[i][j][r];
            }
        }
    }
}

// A 32 x 16 MFMA operand whose rows are channels and whose reduction index runs
// over 16 pixels, from a pixel-major LDS patch of pitch P, by two
// ds_read_b64_tr_b16 (each group of 16 lanes turns 4 pixels x 16 channels into 4
// pixels per lane).  With P = 32 a group pair's rows are 64 consecutive bytes and
// the reads meet no bank twice.
typedef short s16x4 __attribute__((ext_vector_type(4)));
template <int P>
__device__ inline bf16x8 read_tr(const u16* t, int lane) {
    typedef __attribute__((address_space(3))) s16x4 lds4;
    const int L = lane & 15;
    const u16* p = t + (8 * (lane >> 5) + (L >> 2)) * P + 16 * ((lane >> 4) & 1) + 4 * (L & 3);
    const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds4*)p);
    const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds4*)(p + 4 * P));
    typedef short s16x8 __attribute__((ext_vector_type(8)));
    return __builtin_bit_cast(bf16x8, (s16x8)__builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
}

// Weight gradient dw[n][tap*C + c] += sum over pixels of dz[p][n] x[p + tap][c]
// for 32 input channels and 32 output channels (blockIdx.y: pair), every tap:
// nine 32 x 32 accumulators a wave.  A workgroup walks tiles of 8 image rows x 32
// pixels, two rows a wave; the four waves' sums meet in LDS and are added to dw
// with one atomic per weight.  KIND as in k_conv (1: the 64 columns of nine taps
// of four channels in two blocks of 32).
template <int KIND, int MODE>
__global__ __launch_bounds__(256, 2) void k_conv_dw(Img s, const u16* __restrict__ dz, int N, int kp, uint32_t tx,
                                                 uint32_t ty, uint32_t ntiles, int ncb, float* __restrict__ dw) {
    constexpr int TY = 8, HALO = KIND == 0 ? 1 : 0, COLS = TX + 2 * HALO, ROWS = TY + 2 * HALO;
    constexpr int TAPS = KIND == 0 ? 9 : 1, KC = KIND == 1 ? 64 : 32;
    constexpr int PATCH = ROWS * COLS * KC, ZT = TY * TX * 32;
    constexpr int RED = 4 * 1024 * 2;   // one tap's four partial 32 x 32 sums, in u16
    __shared__ __align__(16) u16 t[PATCH + ZT > RED ? PATCH + ZT : RED];
    u16* const z = t + PATCH;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int c0 = (int)(blockIdx.y % ncb) * 32, n0 = (int)(blockIdx.y / ncb) * 32;
    f32x16 acc[TAPS];
#pragma unroll
    for (int k = 0; k < TAPS; ++k)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[k][r] = 0.f;
    for (uint32_t it = blockIdx.x; it < ntiles; it += gridDim.x) {
        const Tile tl = tile_of(it, tx, ty, TY);
        __syncthreads();   // the last tile's reads
        if (KIND == 1) stage_taps<KC, KC, ROWS, 8>(s, tl.b, tl.y0, tl.x0, t);
        else stage<KC, KC, ROWS, COLS, MODE, MODE == IN_ADD ? 4 : 6>(s, tl.b, tl.y0 - HALO, tl.x0 - HALO, c0, t);
        if (KIND == 2) {   // N < 32 columns, the rest zero
#pragma unroll 8
            for (int v = threadIdx.x; v < ZT; v += 256) {
                const int px = v >> 5, n = v & 31, y = tl.y0 + px / TX, x = tl.x0 + px % TX;
                const u16 q = dz[(((size_t)tl.b * s.H + clampi(y, s.H)) * s.W + clampi(x, s.W)) * N + (n < N ? n : 0)];
                z[v] = n < N && y < s.H && x < s.W ? q : (u16)0;
            }
        } else {
            stage_bf<32, 32, TY, TX, 4>(dz, s.H, s.W, N, tl.b, tl.y0, tl.x0, n0, z);
        }
        __syncthreads();
#pragma unroll
        for (int h = 0; h < 4; ++h) {   // two rows of two 16-pixel runs
            const int row = 2 * wave + (h >> 1), x = 16 * (h & 1);
            const bf16x8 b = read_tr<32>(z + (row * TX + x) * 32, lane);
#pragma unroll
            for (int k = 0; k < TAPS; ++k) {
                const int at = KIND == 1 ? (row * COLS + x) * KC + c0 : ((row + k / 3) * COLS + x + k % 3) * KC;
                const bf16x8 a = read_tr<KC>(t + at, lane);
                acc[k] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, acc[k], 0, 0, 0);
            }
        }
    }
    // accumulator register r of lane l: channel 8 (r / 4) + 4 (l / 32) + r % 4, column l % 32
    float* const red = (float*)t;
    const int C = KIND == 1 ? 64 : s.C;
#pragma unroll
    for (int k = 0; k < TAPS; ++k) {
        __syncthreads();
#pragma unroll
        for (int r = 0; r < 16; ++r)
            red[wave * 1024 + (lane & 31) * 32 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3)] = acc[k][r];
        __syncthreads();
        for (int e = threadIdx.x; e < 1024; e += 256) {
            const int n = n0 + (e >> 5), c = c0 + (e & 31);
            const float v = red[e] + red[1024 + e] + red[2048 + e] + red[3072 + e];
            if (n < N && (KIND != 1 || c < 36)) atomicAdd(dw + (size_t)n * kp + k * C + c, v);
        }
    }
}

// dz = g (times y > 0 when relu) as bf16 and its column sums, added to db, four
// channels a thread.  The gradient g of the H x W image is dy itself; or the 2 x 2
// sums of dy at twice the resolution (the adjoint of the upsampling); or dy at half
// the resolution spread over 2 x 2 / 4, plus skip (the adjoint of the pooling, and
// the gradient that came by the skip connection).  Nothing but this pass reads
// such a g, so it is not stored.  N (32, 64 or 128) divides the 1024 values a
// workgroup covers, so a thread keeps its four columns.
//
// Bound by its traffic; with the adjoints in passes of their own the backward of
// 16 images of 512 x 128 spent 1.03 ms on all of them, now 0.63 ms.
enum { GRAD_X = 0, GRAD_UP = 1, GRAD_POOL = 2 };
template <int MODE>
__global__ __launch_bounds__(256) void k_grad_sum(const float* __restrict__ dy, const float* __restrict__ skip,
                                                  const float* __restrict__ y, int relu, uint32_t W, size_t n4, int N,
                                                  u16* __restrict__ dz, float* __restrict__ db) {
    f32x4 s = {0.f, 0.f, 0.f, 0.f};
    const uint32_t n1 = (uint32_t)N / 4;
#pragma unroll 2
    for (size_t e = blockIdx.x * (size_t)256 + threadIdx.x; e < n4; e += (size_t)gridDim.x * 256) {
        f32x4 g;
        if (MODE == GRAD_X) {
            g = *(const f32x4*)(dy + 4 * e);
        } else {   // n4 is below 2^31
            const uint32_t p = (uint32_t)e / n1, c = 4 * ((uint32_t)e - p * n1), row = p / W, x = p - row * W;
            if (MODE == GRAD_UP) {
                const float* q = dy + ((size_t)(2 * row) * (2 * W) + 2 * x) * N + c;
                const size_t down = (size_t)2 * W * N;
                const f32x4 a = *(const f32x4*)q, b = *(const f32x4*)(q + N);
                const f32x4 d = *(const f32x4*)(q + down), f = *(const f32x4*)(q + down + N);
#pragma unroll
                for (int i = 0; i < 4; ++i) g[i] = a[i] + b[i] + d[i] + f[i];
            } else {
                const f32x4 a = *(const f32x4*)(dy + ((size_t)(row >> 1) * (W >> 1) + (x >> 1)) * N + c);
                const f32x4 b = *(const f32x4*)(skip + 4 * e);
#pragma unroll
                for (int i = 0; i < 4; ++i) g[i] = 0.25f * a[i] + b[i];
            }
        }
        if (relu) {
            const f32x4 v = *(const f32x4*)(y + 4 * e);
#pragma unroll
            for (int i = 0; i < 4; ++i) g[i] = v[i] > 0.f ? g[i] : 0.f;
        }
        *(uint2*)(dz + 4 * e) = f2bf4(g);
#pragma unroll
        for (int i = 0; i < 4; ++i) s[i] += g[i];
    }
    __shared__ float red[1024];
#pragma unroll
    for (int i = 0; i < 4; ++i) red[4 * threadIdx.x + i] = s[i];
    __syncthreads();
    if ((int)threadIdx.x < N) {
        float t = 0.f;
        for (int k = threadIdx.x; k < 1024; k += N) t += red[k];
        atomicAdd(db + threadIdx.x, t);
    }
}

// wt[tap][c][n] = w[n][tap*C + c] of up to 16 layers (blockIdx.y), the B operand
// of k_conv_dx.
struct WtLayers {
    int64_t from[16], to[16];
    int cin[16], cout[16], kp[16];
};
__global__ void k_weight_t(const u16* __restrict__ w, WtLayers l, u16* __restrict__ wt) {
    const int k = blockIdx.y, C = l.cin[k], N = l.cout[k], total = 9 * C * N;
    for (int e = blockIdx.x * blockDim.x + threadIdx.x; e < total; e += gridDim.x * blockDim.x) {
        const int tc = e / N, n = e - tc * N;
        wt[l.to[k] + e] = w[l.from[k] + (size_t)n * l.kp[k] + tc];
    }
}

template <int KIND, int KC, int TY, int WM, int WN, int TM, int TN>
hipError_t conv_m(int mode, const Img& s, int Bn, const u16* w, int kp, const float* bias, int relu, int N, float* y,
                  hipStream_t st) {
    const uint32_t tx = (uint32_t)(s.W + TX - 1) / TX, ty = (uint32_t)(s.H + TY - 1) / TY;
    const dim3 grid(tx * ty * (uint32_t)Bn);
    auto go = [&](auto k) { hipLaunchKernelGGL(k, grid, dim3(256), 0, st, s, w, kp, bias, relu, N, tx, ty, y); };
    if constexpr (KIND == 0) {
        if (mode == IN_UP) { go(k_conv<KIND, KC, TY, WM, WN, TM, TN, IN_UP>); return hipGetLastError(); }
        if (mode == IN_ADD) { go(k_conv<KIND, KC, TY, WM, WN, TM, TN, IN_ADD>); return hipGetLastError(); }
    }
    go(k_conv<KIND, KC, TY, WM, WN, TM, TN, IN_X>);
    return hipGetLastError();
}
template <int KC, int TY, int WM, int WN, int TM, int TN>
hipError_t dx_m(const u16* dz, int Bn, int H, int W, const u16* wt, int N, float* dx, hipStream_t st) {
    const uint32_t tx = (uint32_t)(W + TX - 1) / TX, ty = (uint32_t)(H + TY - 1) / TY;
    hipLaunchKernelGGL((k_conv_dx<KC, TY, WM, WN, TM, TN>), dim3(tx * ty * (uint32_t)Bn), dim3(256), 0, st, dz, H, W, wt,
                       N, tx, ty, dx);
    return hipGetLastError();
}

bool aligned16(const void* p) { return ((uintptr_t)p & 15) == 0; }
// what the im2col path refuses (its matrix above 2^31 elements) stays refused
bool fits(int Bn, int H, int W, int kp) { return (uint64_t)Bn * H * W * kp < (1ull << 31); }

}  // namespace

extern "C" {

int nn_conv(const float* x, const float* skip, int mode, int Bn, int H, int W, int cin, int cout, int k, const void* w,
            int kp, const float* bias, int relu, float* y, void* stream) {
    if (Bn < 0 || H < 1 || W < 1 || !fits(Bn, H, W, kp) || kp < cin * k * k || (kp & 7) || !aligned16(w)) return 3;
    if (mode < 0 || mode > 2 || (mode == IN_ADD && !skip) || (mode == IN_UP && ((H | W) & 1))) return 3;
    if (Bn == 0) return 0;
    hipStream_t st = (hipStream_t)stream;
    const Img s{x, skip, H, W, cin};
    const u16* wb = (const u16*)w;
    hipError_t e;
    if (k == 3 && cin == 4 && cout == 32 && kp >= 48 && mode == IN_X)
        e = conv_m<1, 48, 8, 4, 1, 2, 1>(mode, s, Bn, wb, kp, bias, relu, cout, y, st);
    else if (k == 3 && cin == 32 && cout == 32)
        e = conv_m<0, 32, 8, 4, 1, 2, 1>(mode, s, Bn, wb, kp, bias, relu, cout, y, st);
    else if (k == 3 && cin == 32 && cout == 64)
        e = conv_m<0, 32, 8, 4, 1, 2, 2>(mode, s, Bn, wb, kp, bias, relu, cout, y, st);
    else if (k == 3 && cin == 64 && cout == 32)
        e = conv_m<0, 64, 8, 4, 1, 2, 1>(mode, s, Bn, wb, kp, bias, relu, cout, y, st);
    else if (k == 3 && cin == 64 && cout == 64)
        e = conv_m<0, 64, 4, 2, 2, 2, 1>(mode, s, Bn, wb, kp, bias, relu, cout, y, st);
    else if (k == 3 && cin == 64 && cout == 128)
        e = conv_m<0, 64, 4, 2, 2, 2, 2>(mode, s, Bn, wb, kp, bias, relu, cout, y, st);
    else if (k == 3 && cin == 128 && cout == 64)
        e = conv_m<0, 128, 4, 2, 2, 2, 1>(mode, s, Bn, wb, kp, bias, relu, cout, y, st);
    else if (k == 3 && cin == 128 && cout == 128)
        e = conv_m<0, 128, 4, 2, 2, 2, 2>(mode, s, Bn, wb, kp, bias, relu, cout, y, st);
    else if (k == 1 && cin == 32 && cout <= 32 && mode == IN_X)
        e = conv_m<2, 32, 8, 4, 1, 2, 1>(mode, s, Bn, wb, kp, bias, relu, cout, y, st);
    else
        return 3;
    return e == hipSuccess ? 0 : 4;
}

int nn_weight_t(const void* w, int nlayers, const int64_t* from, const int64_t* to, const int* cin, const int* cout,
                const int* kp, void* wt, void* stream) {
    if (nlayers < 0 || nlayers > 16) return 3;
    if (nlayers == 0) return 0;
    WtLayers l{};
    for (int i = 0; i < nlayers; ++i) {
        l.from[i] = from[i]; l.to[i] = to[i];
        l.cin[i] = cin[i]; l.cout[i] = cout[i]; l.kp[i] = kp[i];
    }
    hipLaunchKernelGGL(k_weight_t, dim3(64, nlayers), dim3(256), 0, (hipStream_t)stream, (const u16*)w, l, (u16*)wt);
    return hipGetLastError() == hipSuccess ? 0 : 4;
}

int nn_conv_dx(const void* dz, int Bn, int H, int W, int cin, int cout, const void* wt, float* dx, void* stream) {
    if (Bn < 0 || H < 1 || W < 1 || !fits(Bn, H, W, 9 * cin) || !aligned16(dz) || !aligned16(wt)) return 3;
    if (Bn == 0) return 0;
    hipStream_t st = (hipStream_t)stream;
    const u16 *z = (const u16*)dz, *t = (const u16*)wt;
    hipError_t e;
    if (cout == 32 && cin == 32) e = dx_m<32, 8, 4, 1, 2, 1>(z, Bn, H, W, t, cin, dx, st);
    else if (cout == 32 && cin == 64) e = dx_m<32, 8, 4, 1, 2, 2>(z, Bn, H, W, t, cin, dx, st);
    else if (cout == 64 && cin == 32) e = dx_m<64, 8, 4, 1, 2, 1>(z, Bn, H, W, t, cin, dx, st);
    else if (cout == 64 && cin == 64) e = dx_m<64, 4, 2, 2, 2, 1>(z, Bn, H, W, t, cin, dx, st);
    else if (cout == 64 && cin == 128) e = dx_m<64, 4, 2, 2, 2, 2>(z, Bn, H, W, t, cin, dx, st);
    else if (cout == 128 && cin == 64) e = dx_m<128, 4, 2, 2, 2, 1>(z, Bn, H, W, t, cin, dx, st);
    else if (cout == 128 && cin == 128) e = dx_m<128, 4, 2, 2, 2, 2>(z, Bn, H, W, t, cin, dx, st);
    else return 3;
    return e == hipSuccess ? 0 : 4;
}

int nn_conv_dw(const float* x, const float* skip, int mode, const void* dz, int Bn, int H, int W, int cin, int cout,
               int k, int kp, float* dw, void* stream) {
    if (Bn < 0 || H < 1 || W < 1 || !fits(Bn, H, W, kp) || kp < cin * k * k || !aligned16(dz)) return 3;
    if (mode < 0 || mode > 2 || (mode == IN_ADD && !skip) || (mode == IN_UP && ((H | W) & 1))) return 3;
    const bool taps4 = k == 3 && cin == 4 && cout % 32 == 0 && mode == IN_X, one = k == 1 && cin == 32 && cout <= 32 && mode == IN_X;
    if (!taps4 && !one && !(k == 3 && cin % 32 == 0 && cout % 32 == 0)) return 3;
    if (Bn == 0) return 0;
    const Img s{x, skip, H, W, cin};
    const uint32_t tx = (uint32_t)(W + TX - 1) / TX, ty = (uint32_t)(H + 7) / 8, nt = tx * ty * (uint32_t)Bn;
    const int ncb = taps4 ? 2 : cin / 32, pairs = ncb * ((cout + 31) / 32);
    // two workgroups a CU over all channel pairs (nine accumulators a wave), three
    // where one accumulator leaves the room
    const uint32_t gx = std::max(1u, std::min(nt, (taps4 || one ? 768u : 512u) / (uint32_t)pairs));
    hipStream_t st = (hipStream_t)stream;
    auto go = [&](auto kern) {
        hipLaunchKernelGGL(kern, dim3(gx, pairs), dim3(256), 0, st, s, (const u16*)dz, cout, kp, tx, ty, nt, ncb, dw);
    };
    if (taps4) go(k_conv_dw<1, IN_X>);
    else if (one) go(k_conv_dw<2, IN_X>);
    else if (mode == IN_UP) go(k_conv_dw<0, IN_UP>);
    else if (mode == IN_ADD) go(k_conv_dw<0, IN_ADD>);
    else go(k_conv_dw<0, IN_X>);
    return hipGetLastError() == hipSuccess ? 0 : 4;
}

int nn_grad_sum(const float* dy, const float* skip, int mode, int Bn, int H, int W, const float* y, int relu, int N,
                void* dz, float* db, void* stream) {
    if (Bn < 0 || H < 1 || W < 1 || (N != 32 && N != 64 && N != 128) || !aligned16(dz)) return 3;
    if (mode < 0 || mode > 2 || (mode == GRAD_POOL && (!skip || ((H | W) & 1)))) return 3;
    if (mode != GRAD_X && !fits(Bn, H, W, N)) return 3;
    if (Bn == 0) return 0;
    // 512 workgroups: the column sums' atomics meet on N addresses (the training
    // step's passes over 16 images take 0.63 ms with 512, 0.66 with 1024, 0.84 with
    // 2048 and 256)
    const size_t n4 = (size_t)Bn * H * W * N / 4, blocks = std::min<size_t>(512, (n4 + 255) / 256);
    auto go = [&](auto kern) {
        hipLaunchKernelGGL(kern, dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream, dy, skip, y, relu,
                           (uint32_t)W, n4, N, (u16*)dz, db);
    };
    if (mode == GRAD_UP) go(k_grad_sum<GRAD_UP>);
    else if (mode == GRAD_POOL) go(k_grad_sum<GRAD_POOL>);
    else go(k_grad_sum<GRAD_X>);
    return hipGetLastError() == hipSuccess ? 0 : 4;
}

}  // extern "C"
