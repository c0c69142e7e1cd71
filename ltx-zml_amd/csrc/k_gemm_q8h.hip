// LDS-DMA W8A16 kernels on tiles of 192 rows: ltx_gemm_q8_[bf16_][s32_]{store,
// resid,qkv}_h192 and _store_raw_h192.
#include "gemm_q8.h"

Q8_GEMM_KERNEL(ltx_gemm_q8_store_h192, _Float16, false, LTX_EPI_STORE, false, 3)
Q8_GEMM_KERNEL(ltx_gemm_q8_resid_h192, _Float16, false, LTX_EPI_RESID_GATE, false, 3)
Q8_GEMM_KERNEL(ltx_gemm_q8_qkv_h192, _Float16, false, LTX_EPI_QKV, false, 3)
Q8_GEMM_KERNEL(ltx_gemm_q8_bf16_store_h192, __bf16, false, LTX_EPI_STORE, false, 3)
Q8_GEMM_KERNEL(ltx_gemm_q8_bf16_resid_h192, __bf16, false, LTX_EPI_RESID_GATE, false, 3)
Q8_GEMM_KERNEL(ltx_gemm_q8_bf16_qkv_h192, __bf16, false, LTX_EPI_QKV, false, 3)
Q8_GEMM_KERNEL(ltx_gemm_q8_s32_store_h192, _Float16, true, LTX_EPI_STORE, false, 3)
Q8_GEMM_KERNEL(ltx_gemm_q8_s32_resid_h192, _Float16, true, LTX_EPI_RESID_GATE, false, 3)
Q8_GEMM_KERNEL(ltx_gemm_q8_s32_qkv_h192, _Float16, true, LTX_EPI_QKV, false, 3)
Q8_GEMM_KERNEL(ltx_gemm_q8_bf16_s32_store_h192, __bf16, true, LTX_EPI_STORE, false, 3)
Q8_GEMM_KERNEL(ltx_gemm_q8_bf16_s32_resid_h192, __bf16, true, LTX_EPI_RESID_GATE, false, 3)
Q8_GEMM_KERNEL(ltx_gemm_q8_bf16_s32_qkv_h192, __bf16, true, LTX_EPI_QKV, false, 3)
Q8_GEMM_KERNEL(ltx_gemm_q8_store_raw_h192, _Float16, false, LTX_EPI_STORE, true, 3)
Q8_GEMM_KERNEL(ltx_gemm_q8_bf16_store_raw_h192, __bf16, false, LTX_EPI_STORE, true, 3)
Q8_GEMM_KERNEL(ltx_gemm_q8_s32_store_raw_h192, _Float16, true, LTX_EPI_STORE, true, 3)
Q8_GEMM_KERNEL(ltx_gemm_q8_bf16_s32_store_raw_h192, __bf16, true, LTX_EPI_STORE, true, 3)
