// Four-wave 16-bit GEMMs on tiles of 192 rows:
// ltx_gemm_x4_{f16,bf16}_{store,store_gelu,store32,store32_gelu,resid,qkv}_h192.
#include "gemm_x4.h"

X4_GEMM_KERNEL(ltx_gemm_x4_f16_store_h192, _Float16, LTX_EPI_STORE, 0, 6)
X4_GEMM_KERNEL(ltx_gemm_x4_f16_store_gelu_h192, _Float16, LTX_EPI_STORE, 1, 6)
X4_GEMM_KERNEL(ltx_gemm_x4_f16_store32_h192, _Float16, LTX_EPI_STORE, 2, 6)
X4_GEMM_KERNEL(ltx_gemm_x4_f16_store32_gelu_h192, _Float16, LTX_EPI_STORE, 3, 6)
X4_GEMM_KERNEL(ltx_gemm_x4_f16_resid_h192, _Float16, LTX_EPI_RESID_GATE, 0, 6)
X4_GEMM_KERNEL(ltx_gemm_x4_f16_qkv_h192, _Float16, LTX_EPI_QKV, 0, 6)
X4_GEMM_KERNEL(ltx_gemm_x4_bf16_store_h192, __bf16, LTX_EPI_STORE, 0, 6)
X4_GEMM_KERNEL(ltx_gemm_x4_bf16_store_gelu_h192, __bf16, LTX_EPI_STORE, 1, 6)
X4_GEMM_KERNEL(ltx_gemm_x4_bf16_store32_h192, __bf16, LTX_EPI_STORE, 2, 6)
X4_GEMM_KERNEL(ltx_gemm_x4_bf16_store32_gelu_h192, __bf16, LTX_EPI_STORE, 3, 6)
X4_GEMM_KERNEL(ltx_gemm_x4_bf16_resid_h192, __bf16, LTX_EPI_RESID_GATE, 0, 6)
X4_GEMM_KERNEL(ltx_gemm_x4_bf16_qkv_h192, __bf16, LTX_EPI_QKV, 0, 6)
