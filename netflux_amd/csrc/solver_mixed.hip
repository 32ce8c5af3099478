// Mixed-precision kernels (kernels_mixed.hpp) in their own translation unit,
// compiled with floating-point contraction enabled; the FP64 kernels live in
// solver.hip, compiled without it.
#define NF_DEVICE_HELPERS_ONLY
#define NF_MIXED_KERNELS
#include "kernels_mixed.hpp"

namespace nf {
namespace mx {

hipError_t launch_ghost_mx(bool face, hipStream_t st, const DevMesh &m, const BndArgsMx &a, const float *src) {
    const dim3 g((a.nb + BLOCK - 1) / BLOCK), b(BLOCK);
    if (face) hipLaunchKernelGGL(k_ghost_mx<true>, g, b, 0, st, m, a, src);
    else hipLaunchKernelGGL(k_ghost_mx<false>, g, b, 0, st, m, a, src);
    return hipGetLastError();
}

template <int B, bool FUSE>
static hipError_t sweepA_b(int order, uint32_t ncell, hipStream_t st, const DevMesh &m, const SweepAArgsMx &a) {
    const dim3 g(ncell / B), b(B);
    if (order == 0) hipLaunchKernelGGL((k_sweepA_mx<0, B, FUSE>), g, b, 0, st, m, a);
    else if (order == 1) hipLaunchKernelGGL((k_sweepA_mx<1, B, FUSE>), g, b, 0, st, m, a);
    else hipLaunchKernelGGL((k_sweepA_mx<2, B, FUSE>), g, b, 0, st, m, a);
    return hipGetLastError();
}
template <int B, bool FUSE>
static hipError_t sweepB_b(uint32_t ncell, hipStream_t st, const DevMesh &m, const SweepBArgsMx &a) {
    hipLaunchKernelGGL((k_sweepB_mx<B, FUSE>), dim3(ncell / B), dim3(B), 0, st, m, a);
    return hipGetLastError();
}

hipError_t launch_sweepA_mx(int order, int block, bool fuse, uint32_t ncell, hipStream_t st, const DevMesh &m,
                            const SweepAArgsMx &a) {
    if (block == 128)
        return fuse ? sweepA_b<128, true>(order, ncell, st, m, a) : sweepA_b<128, false>(order, ncell, st, m, a);
    return fuse ? sweepA_b<256, true>(order, ncell, st, m, a) : sweepA_b<256, false>(order, ncell, st, m, a);
}

hipError_t launch_sweepB_mx(int block, bool fuse, uint32_t ncell, hipStream_t st, const DevMesh &m,
                            const SweepBArgsMx &a) {
    if (block == 128) return fuse ? sweepB_b<128, true>(ncell, st, m, a) : sweepB_b<128, false>(ncell, st, m, a);
    return fuse ? sweepB_b<256, true>(ncell, st, m, a) : sweepB_b<256, false>(ncell, st, m, a);
}

hipError_t launch_prim_mx(dim3 g, hipStream_t st, const double *U, float *V, uint32_t N) {
    hipLaunchKernelGGL(k_prim_mx, g, dim3(BLOCK), 0, st, U, V, N);
    return hipGetLastError();
}

hipError_t launch_apply_mx(dim3 g, hipStream_t st, const DevMesh &m, const ApplyArgs &a) {
    hipLaunchKernelGGL(k_apply_mx, g, dim3(BLOCK), 0, st, m, a);
    return hipGetLastError();
}

}  // namespace mx
}  // namespace nf
