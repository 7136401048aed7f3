// Several D2Q9 steps per launch.
//
// A single step of a 2D lattice is bound by its launch (256 x 64: 5.9 us for 16 k
// nodes) or by the caches (1021 x 256 FP32: 7.9 us, 4 us of copy), not by its
// arithmetic.  Here a workgroup takes a square of 32 x 32 nodes, one a thread,
// pulls the post-collision populations of the square once, advances them `steps`
// steps with the streamed populations in LDS and writes the inner nodes: after
// step s the nodes s from the rim are still exact, so a frame of `steps`
// nodes is recomputed by the neighbouring squares instead of being exchanged.
// The node update is the step's own (walls, Zou-He faces, moments, collision), so
// the bits are too.
//
// Per step, one launch a step / several (the number): FP64 256 x 64 5.73 / 2.01 us
// (12), 1021 x 256 10.7 / 6.0 (4), 4096 x 1024 113 / 73 (4); FP32 5.37 / 1.47,
// 8.0 / 3.7, 78 / 33.  What bounds it: on few squares the launch and the chain of
// LDS round trips (about 1.3 us a step FP64), on many the instructions of the node
// update, 1.8 times with the frame of 4.
#include "lbm_square.h"

namespace lbm {

// FULL: more squares than CUs; FP32 then keeps to 64 registers so that two
// workgroups share a CU (4096 x 1024: 52.7 -> 33.1 us per step; with one square a
// CU the tighter code only costs, 256 x 64 1.47 -> 1.57 us).
template <int S, int C, bool FULL>
__global__ __launch_bounds__(kSquare, S == 1 && FULL ? 8 : 4) void k_multi2(const typename Io<D2Q9, S>::raw* __restrict__ src,
                                                   typename Io<D2Q9, S>::raw* __restrict__ dst,
                                                   const uint32_t* __restrict__ node,
                                                   const uint32_t* __restrict__ cidx, KParams kp, Fields fl, int steps,
                                                   uint32_t tx) {
    using L = D2Q9;
    using T = typename Io<L, S>::T;
    __shared__ T lds[8][kSquare];
    const int tid = threadIdx.x, lx = tid & (kSide - 1), ly = tid / kSide;
    const int in = kSide - 2 * steps, nx = kp.nx, ny = kp.ny;
    const uint32_t b = xcd_block(blockIdx.x, gridDim.x, kp.xcd_shift, kp.xchunk_shift), by = b / tx;
    const int ux = (int)(b - by * tx) * in - steps + lx, uy = (int)by * in - steps + ly;
    // periodic axes wrap (boxes smaller than the frame too)
    int x = ux, y = uy;
    if (kp.per[0]) { x %= nx; x = x < 0 ? x + nx : x; }
    if (kp.per[1]) { y %= ny; y = y < 0 ? y + ny : y; }
    uint32_t idx = 0, own = kNone, nd = 0;
    if (x >= 0 && x < nx && y >= 0 && y < ny) {
        idx = (uint32_t)y * (uint32_t)nx + (uint32_t)x;
        own = cidx[idx];
        nd = node[idx];
    }
    const bool live = own != kNone;
    T p[L::Q];   // the node's post-collision populations
#pragma unroll
    for (int i = 0; i < L::Q; ++i) p[i] = live ? Io<L, S>::ld(src, tslot<L>(i, own), i) : (T)0;
    const uint2 ln = square_links(nd, !kp.per[0] && x == 0, !kp.per[0] && x == nx - 1, !kp.per[1] && y == 0,
                                  !kp.per[1] && y == ny - 1);
    double ub[2] = {0.0, 0.0};   // the face velocity, read once
    if (live && (nd >> kClsShift) != FLUID && fl.ubc) { ub[0] = fl.ubc[idx]; ub[1] = fl.vbc[idx]; }
    Fields fn = fl;
    fn.ubc = ub;
    fn.vbc = ub + 1;
    square_steps<T, C>(kp, fn, idx, live, nd, ln.x, ln.y, steps, lds, p);
    const int rim = min(min(lx, kSide - 1 - lx), min(ly, kSide - 1 - ly));
    if (live && rim >= steps && ux < nx && uy < ny) {   // ux, uy >= 0 inside the frame
#pragma unroll
        for (int i = 0; i < L::Q; ++i) sto(dst, tslot<L>(i, own), Io<L, S>::pk(p[i], i));
    }
}

template <int S, int C>
static hipError_t multi_t(const KParams& kp, const void* src, void* dst, const uint32_t* node, const uint32_t* cidx,
                          const Fields& fl, int steps, hipStream_t st) {
    using raw = typename Io<D2Q9, S>::raw;
    const int in = kSide - 2 * steps;
    const uint32_t tx = (uint32_t)(kp.nx + in - 1) / in, ty = (uint32_t)(kp.ny + in - 1) / in;
    auto go = [&](auto k) {
        hipLaunchKernelGGL(k, dim3(tx * ty), dim3(kSquare), 0, st, (const raw*)src, (raw*)dst, node, cidx, kp, fl, steps,
                           tx);
    };
    if (S == 1 && tx * ty > 256) go(k_multi2<S, C, true>);
    else go(k_multi2<S, C, false>);
    return hipGetLastError();
}

hipError_t launch_multi2(int storage, int collision, const KParams& kp, const void* src, void* dst,
                         const uint32_t* node, const uint32_t* cidx, const Fields& fl, int steps, hipStream_t st) {
    if (steps < 1 || 2 * steps >= kSide || storage > 1) return hipErrorInvalidValue;
    if (storage == 0) {
        switch (collision) {
        case 0: return multi_t<0, 0>(kp, src, dst, node, cidx, fl, steps, st);
        case 1: return multi_t<0, 1>(kp, src, dst, node, cidx, fl, steps, st);
        default: return multi_t<0, 2>(kp, src, dst, node, cidx, fl, steps, st);
        }
    }
    switch (collision) {
    case 0: return multi_t<1, 0>(kp, src, dst, node, cidx, fl, steps, st);
    case 1: return multi_t<1, 1>(kp, src, dst, node, cidx, fl, steps, st);
    default: return multi_t<1, 2>(kp, src, dst, node, cidx, fl, steps, st);
    }
}

}  // namespace lbm
