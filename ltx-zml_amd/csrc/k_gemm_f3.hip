// f32 GEMMs on bf16 MFMAs (128 x 128 tiles, four waves):
// ltx_gemm_f3_{i8f32,i8f16,w16}_{store,store_gelu,resid}, and the exact split
// of their f32 activations into three bf16 planes.
#include "gemm_f3.h"

// The split of A (split3, ltx_device.h). Bandwidth-bound: 32 B in and 48 B out
// a thread.
extern "C" __global__ void __launch_bounds__(256) ltx_split3(const LtxSplit3Args a) {
    const size_t i = ((size_t)blockIdx.x * 256 + threadIdx.x) * 8;
    if (i >= a.n) return;
    const f32x4 x0 = *(const f32x4*)(a.x + i), x1 = *(const f32x4*)(a.x + i + 4);
    u32x4 p[3];
    split3({x0[0], x0[1], x0[2], x0[3], x1[0], x1[1], x1[2], x1[3]}, p);
    *(u32x4*)(a.p0 + i) = p[0];
    *(u32x4*)(a.p1 + i) = p[1];
    *(u32x4*)(a.p2 + i) = p[2];
}

F3_GEMM_KERNEL(ltx_gemm_f3_i8f32_store, LTX_B_I8_F32S, LTX_EPI_STORE, 2)
F3_GEMM_KERNEL(ltx_gemm_f3_i8f32_store_gelu, LTX_B_I8_F32S, LTX_EPI_STORE, 3)
F3_GEMM_KERNEL(ltx_gemm_f3_i8f32_resid, LTX_B_I8_F32S, LTX_EPI_RESID_GATE, 0)
F3_GEMM_KERNEL(ltx_gemm_f3_i8f16_store, LTX_B_I8_F16S, LTX_EPI_STORE, 2)
F3_GEMM_KERNEL(ltx_gemm_f3_i8f16_store_gelu, LTX_B_I8_F16S, LTX_EPI_STORE, 3)
F3_GEMM_KERNEL(ltx_gemm_f3_i8f16_resid, LTX_B_I8_F16S, LTX_EPI_RESID_GATE, 0)
F3_GEMM_KERNEL(ltx_gemm_f3_w16_store, LTX_B_W16, LTX_EPI_STORE, 2)
F3_GEMM_KERNEL(ltx_gemm_f3_w16_store_gelu, LTX_B_W16, LTX_EPI_STORE, 3)
F3_GEMM_KERNEL(ltx_gemm_f3_w16_resid, LTX_B_W16, LTX_EPI_RESID_GATE, 0)
