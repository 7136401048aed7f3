// 3D nodes whose closure the step of every node leaves out: extrapolating
// outlets and curved walls.
#include "lbm_step.h"

namespace lbm {

// The nodes of kp.edge: runs after k_step has updated every node without these
// closures, and overwrites them.
template <class L, int S, int C>
__global__ __launch_bounds__(64) void k_edge(const typename Io<L, S>::raw* __restrict__ src,
                                             typename Io<L, S>::raw* __restrict__ dst,
                                             const uint32_t* __restrict__ didx,
                                             const uint32_t* __restrict__ nodew,
                                             const uint32_t* __restrict__ cidx, KParams kp, Fields fl,
                                             int write_macros) {
    const uint32_t t = blockIdx.x * 64u + threadIdx.x;
    if (t >= kp.nedge) return;
    step_node<L, S, C, true, true, true, true>(src, dst, didx, nodew, cidx, kp, fl, write_macros, kp.edge[t]);
}

template <int S, int C>
static hipError_t edge_t(const KParams& kp, const void* src, void* dst, const uint32_t* cidx, const Fields& fl, int wm,
                         hipStream_t st) {
    using raw = typename Io<D3Q19, S>::raw;
    hipLaunchKernelGGL((k_edge<D3Q19, S, C>), dim3((kp.nedge + 63) / 64), dim3(64), 0, st, (const raw*)src, (raw*)dst,
                       kp.didx, kp.nodew, cidx, kp, fl, wm);
    return hipGetLastError();
}
template <int S>
static hipError_t edge_c(int c, const KParams& kp, const void* src, void* dst, const uint32_t* cidx, const Fields& fl,
                         int wm, hipStream_t st) {
    switch (c) {
    case 0: return edge_t<S, 0>(kp, src, dst, cidx, fl, wm, st);
    case 1: return edge_t<S, 1>(kp, src, dst, cidx, fl, wm, st);
    default: return edge_t<S, 2>(kp, src, dst, cidx, fl, wm, st);
    }
}
hipError_t launch_edge(int s, int c, const KParams& kp, const void* src, void* dst, const uint32_t* cidx,
                       const Fields& fl, bool wm, hipStream_t st) {
    switch (s) {
    case 0: return edge_c<0>(c, kp, src, dst, cidx, fl, wm ? 1 : 0, st);
    case 1: return edge_c<1>(c, kp, src, dst, cidx, fl, wm ? 1 : 0, st);
    case 2: return edge_c<2>(c, kp, src, dst, cidx, fl, wm ? 1 : 0, st);
    default: return edge_c<3>(c, kp, src, dst, cidx, fl, wm ? 1 : 0, st);
    }
}

}  // namespace lbm
