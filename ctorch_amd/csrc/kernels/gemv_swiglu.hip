// Projection kernels with the SWIGLU epilogue: the GEMV (one activation row) and the matrix-core variant.
#include "kernels/gemm_f32.h"
#include "kernels/gemm_mid.h"

dlk::gemv::Kernel dlk_gemv_kernel_swiglu(const dlk_gemv_params& p, int mt) {
    return dlk::gemv::resolve<DLK_EPI_SWIGLU>(p, mt);
}

dlk::gemv::Kernel dlk_gemm_kernel_swiglu(const dlk_gemv_params& p, int mt, int nc) {
    return dlk::gemm::resolve<DLK_EPI_SWIGLU>(p, mt, nc);
}

dlk::gemv::Kernel dlk_gemm_reduce_swiglu(const dlk_gemv_params& p) {
    return dlk::gemm::resolve_reduce<DLK_EPI_SWIGLU>(p);
}

dlk::gemv::Kernel dlk_tiles_kernel_swiglu(const dlk_gemv_params& p) {
    return dlk::tiles::resolve<DLK_EPI_SWIGLU>(p);
}

const void* dlk_gemm_f32_kernel_swiglu(const dlk_gemv_params& p, int shape) {
    return dlk::gemm32::resolve<DLK_EPI_SWIGLU>(p, shape);
}

const void* dlk_mid_kernel_swiglu(const dlk_gemv_params& p) {
    return dlk::mid::resolve<DLK_EPI_SWIGLU>(p);
}
