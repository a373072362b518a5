// Projection kernels with the QKV epilogue: the GEMV (one activation row) and the matrix-core variant.
#include "kernels/gemm_f32.h"
#include "kernels/gemm_mid.h"

dlk::gemv::Kernel dlk_gemv_kernel_qkv(const dlk_gemv_params& p, int mt) {
    return dlk::gemv::resolve<DLK_EPI_QKV>(p, mt);
}

dlk::gemv::Kernel dlk_gemm_kernel_qkv(const dlk_gemv_params& p, int mt, int nc) {
    return dlk::gemm::resolve<DLK_EPI_QKV>(p, mt, nc);
}

dlk::gemv::Kernel dlk_gemm_reduce_qkv(const dlk_gemv_params& p) {
    return dlk::gemm::resolve_reduce<DLK_EPI_QKV>(p);
}

dlk::gemv::Kernel dlk_tiles_kernel_qkv(const dlk_gemv_params& p) {
    return dlk::tiles::resolve<DLK_EPI_QKV>(p);
}

const void* dlk_gemm_f32_kernel_qkv(const dlk_gemv_params& p, int shape) {
    return dlk::gemm32::resolve<DLK_EPI_QKV>(p, shape);
}

const void* dlk_mid_kernel_qkv(const dlk_gemv_params& p) {
    return dlk::mid::resolve<DLK_EPI_QKV>(p);
}
