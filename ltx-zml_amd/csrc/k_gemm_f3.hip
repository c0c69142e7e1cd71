// f32 GEMMs on bf16 MFMAs (128 x 128 tiles, four waves):
// ltx_gemm_f3_{i8f32,i8f16,w16}_{store,store_gelu,resid}, and the exact split
// of their f32 activations into three bf16 planes.
#include "gemm_f3.h"

// x = p0 + p1 + p2: p0 the bits of x down to the eighth significant one, p1
// the same of the rest, p2 what is left (at most 8 significant bits: exact).
// An infinity is its own first plane with nothing left (inf - inf would leave
// a NaN); a NaN leaves one in the second plane. Bandwidth-bound: 32 B in and
// 48 B out a thread.
extern "C" __global__ void __launch_bounds__(256) ltx_split3(const LtxSplit3Args a) {
    const size_t i = ((size_t)blockIdx.x * 256 + threadIdx.x) * 8;
    if (i >= a.n) return;
    const f32x4 x0 = *(const f32x4*)(a.x + i), x1 = *(const f32x4*)(a.x + i + 4);
    uint32_t h[8], m[8], l[8];
#pragma unroll
    for (int e = 0; e < 8; e++) {
        const float x = e < 4 ? x0[e & 3] : x1[e & 3];
        h[e] = __builtin_bit_cast(uint32_t, x) & 0xffff0000u;
        const float r = __builtin_isinf(x) ? 0.0f : x - __builtin_bit_cast(float, h[e]);
        m[e] = __builtin_bit_cast(uint32_t, r) & 0xffff0000u;
        l[e] = __builtin_bit_cast(uint32_t, r - __builtin_bit_cast(float, m[e]));
    }
    // the upper halves of a pair
    auto pk = [](uint32_t lo, uint32_t hi) { return __builtin_amdgcn_perm(hi, lo, 0x07060302u); };
    *(u32x4*)(a.p0 + i) = u32x4{pk(h[0], h[1]), pk(h[2], h[3]), pk(h[4], h[5]), pk(h[6], h[7])};
    *(u32x4*)(a.p1 + i) = u32x4{pk(m[0], m[1]), pk(m[2], m[3]), pk(m[4], m[5]), pk(m[6], m[7])};
    *(u32x4*)(a.p2 + i) = u32x4{pk(l[0], l[1]), pk(l[2], l[3]), pk(l[4], l[5]), pk(l[6], l[7])};
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
