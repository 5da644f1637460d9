// Instantiations and launch of the register-staged GEMM (pe_gemm_rs.h).
#include "pe_gemm_rs.h"

namespace pe {

template <typename E, int BM, int BN, int BK, int MINB>
static const void* rs_kernel_ab(int al, int bl) {
    if (al == L_MN)
        return bl == L_MN ? reinterpret_cast<const void*>(&gemm_rs_kernel<E, BM, BN, BK, L_MN, L_MN, MINB>)
                          : reinterpret_cast<const void*>(&gemm_rs_kernel<E, BM, BN, BK, L_MN, L_K, MINB>);
    return bl == L_MN ? reinterpret_cast<const void*>(&gemm_rs_kernel<E, BM, BN, BK, L_K, L_MN, MINB>)
                      : reinterpret_cast<const void*>(&gemm_rs_kernel<E, BM, BN, BK, L_K, L_K, MINB>);
}

// float32: 128x128 tiles, 16-k slabs, 48 KB of LDS, two blocks per CU.  float16:
// 128x128 tiles with 64-k slabs (64 KB, two blocks per CU; 32-k slabs at three
// blocks per CU: 2001 x 1537 x 3003 53.5 us against 50.0), 64x64 with 32-k ones
// (20 x 201 x 99 x 303 10.4 us, 64-k 11.5; both before DlOperand's 64-row
// fragment offsets were computed, 8.6 since).
static const void* rs_kernel(int dtype, int tile, int al, int bl) {
    if (dtype == PE_F32) return rs_kernel_ab<F32, 128, 128, 16, 2>(al, bl);
    return tile == 128 ? rs_kernel_ab<F16, 128, 128, 64, 2>(al, bl) : rs_kernel_ab<F16, 64, 64, 32, 4>(al, bl);
}

hipError_t launch_gemm_rs(int dtype, int tile, int al, int bl, const GemmArgs& g, hipStream_t s) {
    if (dtype == PE_F32 && tile != 128) return hipErrorInvalidConfiguration;
    GemmArgs a = g;
    if (a.grid > kMaxBlocks) a.grid = uint32_t(kMaxBlocks);  // the tile walk strides over the rest
    void* args[] = {&a};
    return hipLaunchKernel(rs_kernel(dtype, tile, al, bl), dim3(a.grid), dim3(kGemmThreads), args, 0, s);
}

}  // namespace pe
