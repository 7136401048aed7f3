// One node's update in the step kernels that take a node list (lbm_kernels.hip,
// lbm_edge.hip): pull, walls and faces, moments, collision, store.
#pragma once
#include "lbm_device.h"

namespace lbm {

// Store of one node's post-collision populations.  The 16-bit storages use
// stochastic rounding (unbiased: a body force smaller than half an ulp of the
// stored deviation still accumulates), with random bits from a hash of the
// compact node index and a per-launch seed, rotated per direction; results are
// deterministic for a given seed sequence.
// LAY: the buffer's layout, 0 tested at run time (kp.tile), 1 known to be
// tiles, 2 known to be SoA planes.
// X: out holds the stored values x_i = h_i / a_i of a 16-bit storage (no
// scaling before the conversion).
template <class L, int S, int LAY = 0, bool X = false>
__device__ inline void store_node(typename Io<L, S>::raw* __restrict__ dst, const KParams& kp, uint32_t own,
                                  const typename Io<L, S>::T* out) {
    using raw = typename Io<L, S>::raw;
    // With the tile layout a node's populations are 64 elements apart: one
    // 64-bit base, and each store's offset is a constant (an immediate of the
    // store instruction rather than an add per population).  With known SoA
    // planes each plane has its own (uniform) base and every store the same
    // offset, the node's index.
    raw* const tb = LAY == 1 ? (raw*)((char*)dst + (size_t)tslot<L>(0, own) * sizeof(raw)) : dst;
    auto base = [&](int i) { return LAY == 1 ? tb : LAY == 2 ? dst + (size_t)i * kp.qstride : dst; };
    auto slot = [&](int i) { return LAY == 1 ? 64u * (uint32_t)i : LAY == 2 ? own : paddr<L>(kp, i, own); };
    if constexpr (S >= 2) {
        if (kp.sr) {
            uint32_t h = own * 0x9E3779B1u + kp.seed;
            h ^= h >> 15;
            h *= 0x2C1B3C6Du;
            h ^= h >> 12;
            // the conversions write the low half of one register in turn (no
            // register to clear per population)
            typename Io<L, S>::pair acc = {0, 0};
#pragma unroll
            for (int i = 0; i < L::Q; ++i) {
                const uint32_t rnd = (h << (i & 31)) | (h >> ((32 - i) & 31));
                if constexpr (X) acc = Io<L, S>::srx(acc, out[i], rnd);
                else acc = Io<L, S>::sr(acc, out[i], i, rnd);
                sto(base(i), slot(i), (raw)acc[0]);
            }
            return;
        }
    }
#pragma unroll
    for (int i = 0; i < L::Q; ++i) {
        if constexpr (X) sto(base(i), slot(i), Io<L, S>::px(out[i]));
        else sto(base(i), slot(i), Io<L, S>::pk(out[i], i));
    }
}

// One step of compact node own: pull, walls and faces, moments, collision, store.
// HH, CURVED, EXT as in post_boundary.
template <class L, int S, int C, bool OPEN, bool HH = true, bool CURVED = true, bool EXT = true>
__device__ inline void step_node(const typename Io<L, S>::raw* __restrict__ src,
                                 typename Io<L, S>::raw* __restrict__ dst, const uint32_t* __restrict__ didx,
                                 const uint32_t* __restrict__ nodew, const uint32_t* __restrict__ cidx,
                                 const KParams& kp, const Fields& fl, int write_macros, uint32_t own) {
    using T = typename Io<L, S>::T;
    const uint32_t idx = didx[own];
    const uint32_t nd = nodew[own];
    const uint32_t q1 = fdiv(idx, kp.mx, kp.sx);
    const int x = (int)(idx - q1 * (uint32_t)kp.nx);
    const uint32_t zq = fdiv(q1, kp.my, kp.sy);
    const int y = (int)(q1 - zq * (uint32_t)kp.ny), z = (int)zq;
    const uint32_t cls = nd >> kClsShift;
    T h[L::Q];
    post_boundary<L, S, OPEN, false, HH, CURVED, EXT>(src, kp, fl, nodew, cidx, own, nd, x, y, z, idx, h);
    T drho, rho, u[3];
    moments<L, T>(kp, cls, h, drho, rho, u);
    if (OPEN) frozen_macros<T>(kp, fl, cls, idx, drho, rho, u);
    if (write_macros) {
        fl.rho[idx] = (double)rho; fl.u[idx] = (double)u[0];
        fl.v[idx] = (double)u[1]; fl.w[idx] = (double)u[2];
    }
    if (OPEN && L::Q == 19 && fl.om_out && is_outlet3(cls)) {
        const size_t n = (size_t)kp.nx * kp.ny * kp.nz;
        fl.om_out[idx] = (double)rho; fl.om_out[n + idx] = (double)u[0];
        fl.om_out[2 * n + idx] = (double)u[1]; fl.om_out[3 * n + idx] = (double)u[2];
    }
    T out[L::Q];
    collide<L, T, C>(kp, h, drho, rho, u, out);
    store_node<L, S>(dst, kp, own, out);
}

}  // namespace lbm
