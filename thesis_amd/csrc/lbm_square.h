// Several steps of a square of 32 x 32 D2Q9 nodes in LDS, shared by the
// single-lattice kernel (lbm_multi2.hip) and the batch (lbm_batch.hip).
#pragma once
#include "lbm_device.h"

namespace lbm {

constexpr int kSide = 32, kSquare = kSide * kSide;   // nodes a side, threads a workgroup

// Directions of node word nd whose source is beyond a wall (x), or beyond a
// non-periodic face given by the flags (y).
__device__ __forceinline__ uint2 square_links(uint32_t nd, bool xl, bool xh, bool yl, bool yh) {
    using L = D2Q9;
    uint32_t wall = 0, face = 0;
#pragma unroll
    for (int i = 1; i < L::Q; ++i) {
        if ((nd >> L::opp(i)) & 1u) wall |= 1u << i;
        if ((L::cx(i) > 0 && xl) || (L::cx(i) < 0 && xh) || (L::cy(i) > 0 && yl) || (L::cy(i) < 0 && yh)) face |= 1u << i;
    }
    return make_uint2(wall, face & ~wall);
}

// Advances the square's nodes, one a thread with post-collision populations p,
// by `steps` steps; after step s the nodes with rim >= s (distance from the
// square's edge) are exact.  lds: populations 1..8 (the rest population stays with
// its thread).  fn.ubc, fn.vbc: this node's face velocity (one value each), idx its
// place in fn.frz.
template <class T, int C>
__device__ __forceinline__ void square_steps(const KParams& kp, const Fields& fn, size_t idx, bool live, uint32_t nd,
                                    uint32_t wall, uint32_t out, int steps, T (&lds)[8][kSquare], T (&p)[9]) {
    using L = D2Q9;
    const int tid = threadIdx.x, lx = tid & (kSide - 1), ly = tid / kSide;
    const uint32_t cls = nd >> kClsShift;
    const bool half = kp.wall == 0;
    const uint32_t links = __any((wall | out) != 0);   // uniform: whether any node of the wave has such a link
    const int rim = min(min(lx, kSide - 1 - lx), min(ly, kSide - 1 - ly));
#pragma unroll
    for (int i = 1; i < L::Q; ++i) lds[i - 1][tid] = p[i];
    for (int s = 1; s <= steps; ++s) {
        const bool on = live && rim >= s;
        T h[L::Q];
        __syncthreads();
        if (on) {
            h[0] = p[0];
#pragma unroll
            for (int i = 1; i < L::Q; ++i) {
                h[i] = lds[i - 1][tid - L::cx(i) - kSide * L::cy(i)];
            }
            if (links) {
#pragma unroll
                for (int i = 1; i < L::Q; ++i) {
                    const T w = half ? p[L::opp(i)] : p[i];
                    h[i] = (wall >> i) & 1u ? w : ((out >> i) & 1u ? p[i] : h[i]);
                }
            }
        }
        __syncthreads();
        if (on) {
            if (cls != FLUID || links) {
                if (cls == VEL_W) zou_inlet<L, T>(kp, fn, 0, nd, h);
                if (cls == VEL_N) zou_lid<L, T>(kp, fn, 0, nd, h);
                if (kp.wall == 1 && (nd & kBBMask)) onnode_walls<L, T>(nd, h);
                if (cls == PRES_E) zou_outlet<L, T>(kp, fn, 0, h);
            }
            T drho, rho, u[3];
            moments<L, T>(kp, cls, h, drho, rho, u);
            frozen_macros<T>(kp, fn, cls, idx, drho, rho, u);
            collide<L, T, C>(kp, h, drho, rho, u, p);
#pragma unroll
            for (int i = 1; i < L::Q; ++i) lds[i - 1][tid] = p[i];
        }
    }
}

}  // namespace lbm
