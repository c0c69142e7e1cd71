// f32 GEMM on bf16 MFMAs for gfx950: y[M][N] = A[M][K] . W[N][K]^T, A f32, W
// int8 with one scale per 128 consecutive k (ltx/block.zig:462-471) or bf16.
//
// The f32 MFMA runs at 1/16 of the bf16 MFMA's rate (157 against 2,500 TFLOP/s
// at the quoted clock). Three bf16 products carry an f32 one without losing a
// bit: an f32 is the exact sum of three bf16 (a0 its leading 8 significant
// bits, a1 the next 8, a2 the last 8: ltx_split3), an int8 weight is a bf16,
// and a bf16 x bf16 product is exact in f32. So
//   sum_k a q = sum_k a0 q + sum_k a1 q + sum_k a2 q
// takes three MFMAs of 16x16x32 with f32 accumulation. The scale is applied in
// f32 to the sum of each group of 128 k, y += s P, where the f32 MFMA kernel
// rounds f32(q) s for every weight; a bf16 weight needs no scale. Fewer
// roundings than the f32 MFMA's chain (12 MFMA sums a group and one fma,
// against 32 MFMA sums of four products): at 1,024 x 12,288 x 4,096 the error
// against 64 bits is 1.6e-7 instead of 1.1e-6, a block's 2.5e-7 instead of
// 1.8e-6. The product there takes 268 us + 8 us for the split (1.15 PFLOP/s
// of bf16 MFMAs: bound by the matrix cores) instead of 835 us (124 TFLOP/s).
//
// Workgroup: 4 waves, one per SIMD, output tile 128 x 128, each wave 64 x 64 as
// 4 x 4 blocks of 16 x 16; its 64 accumulators and, with scales, the group's 64
// partial sums. K in tiles of 64 through LDS by LDS DMA into two stages: the
// three planes of A (16 KB each) and W as stored (int8 8 KB, bf16 16 KB), in the
// layout and swizzles of gemm_s4.h. The schedule is that of gemm_x4.h: one
// barrier a tile, entered with the tile's second step in registers; each step
// of 32 k is 48 MFMAs with the 16 fragment reads of the next step between them,
// and the DMA two tiles ahead in the first step after the barrier. W fragments
// are converted (int8 -> f32 -> the upper half, exact) between the MFMAs of the
// step before the one that uses them. A group's partial sums are folded into
// the accumulators between the first 16 MFMAs of the next group, which restart
// them from zero.
//
// A group's sum of a q may leave f32's range (from |a| = 2^114 on) where y does
// not. A tile with a sum that is not finite is therefore formed once more with
// the int8 weights times 2^-14 and the scales times 2^14 (exact): the range is
// that of A and y, and an infinity or NaN in A stays one. Doing so always cost
// 8 % (one subtraction for two weights: the VALU has no room beside these
// MFMAs). At the other end the lowest plane ends at bf16's smallest subnormal:
// values keep all of their bits from 2^-110 on.
#pragma once
#include "gemm_s4.h"

__shared__ __attribute__((aligned(1024))) uint8_t f3q_st0[57344];
__shared__ __attribute__((aligned(1024))) uint8_t f3q_st1[57344];
__shared__ __attribute__((aligned(1024))) uint8_t f3w_st0[65536];
__shared__ __attribute__((aligned(1024))) uint8_t f3w_st1[65536];
__shared__ int f3_redo;  // 1 + the tile (and slice) to form once more

template <bool Q, int S>
__device__ __forceinline__ uint8_t* f3_stage() {
    if constexpr (Q)
        return S == 0 ? f3q_st0 : f3q_st1;
    else
        return S == 0 ? f3w_st0 : f3w_st1;
}

template <int BK, int EPI, int SF>
struct F3Gemm {
    static constexpr bool Q = BK != LTX_B_W16;
    static constexpr int NDB = Q ? 2 : 4;  // W DMA instructions per wave and tile (A: 12)
    static constexpr int WOFF = 49152;     // W within a stage
    typedef typename std::conditional<Q, u32x2, u32x4>::type WF;  // a W fragment as read from LDS
    const LtxGemmArgs& a;
    f32x4 acc[4][4];
    f32x4 P[Q ? 4 : 1][4];  // the running group's partial sums
    __amdgpu_buffer_rsrc_t ra_[3], rb_;
    uint32_t ga[4], gb[4];      // per-lane DMA source offsets, K-tile 0 of the slice
    int la, lb;                 // this wave's DMA destinations within a stage (A plane, W)
    uint32_t offa[2], offb[2];  // fragment reads of step s (block i adds 2048 i; int8 W 1024 i)
    uint32_t wx;                // XOR that makes the weight bytes two's complement
    const char* sc;             // the lane's scale of column block 0, first group of the slice
    float s[4];                 // scales of the lane's columns, current group
    u32x4 fa0[12], fa1[12];     // A fragments (plane p, block i: 4 p + i) of steps 0 and 1
    bf16x8 fb0[4], fb1[4];      // W operands

    __device__ __forceinline__ F3Gemm(const LtxGemmArgs& args) : a(args) {}

    // DMA instruction d of K-tile kt into stage S: A (plane d / 4), then W
    template <int S>
    __device__ __forceinline__ void dma1(int d, int kt) {
        if (d < 12)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(ra_[d >> 2],
                                                     (lds_vptr)(f3_stage<Q, S>() + la + 16384 * (d >> 2) + 1024 * (d & 3)),
                                                     16, ga[d & 3], kt * 128, 0, 0);
        else
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rb_, (lds_vptr)(f3_stage<Q, S>() + lb + 1024 * (d - 12)), 16,
                                                     gb[d - 12], kt * (Q ? 64 : 128), 0, 0);
    }
    template <int S>
    __device__ __forceinline__ void dma(int kt) {
#pragma unroll
        for (int d = 0; d < 12 + NDB; d++) dma1<S>(d, kt);
    }

    template <int S, int STEP>
    __device__ __forceinline__ WF read_w(int j) {
        return *(const WF*)(f3_stage<Q, S>() + offb[STEP] + (Q ? 1024 : 2048) * j);
    }
    template <int S, int STEP>
    __device__ __forceinline__ u32x4 read_a(int i) {
        return *(const u32x4*)(f3_stage<Q, S>() + offa[STEP] + 16384 * (i >> 2) + 2048 * (i & 3));
    }

    // 8 weights as a bf16 operand: an int8 is exact in the upper half of its f32.
    // X: times 2^-14, 14 off the exponents of a pair (a zero's stays zero: the
    // subtraction saturates).
    template <bool X>
    __device__ __forceinline__ bf16x8 operand(const WF& w) {
        if constexpr (Q) {
            u32x4 o;
#pragma unroll
            for (int d = 0; d < 2; d++) {
                const uint32_t x = w[d] ^ wx;
#pragma unroll
                for (int e = 0; e < 2; e++) {
                    const float lo = (float)(int8_t)(x >> (16 * e)), hi = (float)(int8_t)(x >> (16 * e + 8));
                    uint32_t b = __builtin_amdgcn_perm(__builtin_bit_cast(uint32_t, hi),
                                                       __builtin_bit_cast(uint32_t, lo), 0x07060302u);
                    if (X) {
                        const u16x2 m = __builtin_elementwise_sub_sat(__builtin_bit_cast(u16x2, b), (u16x2)(14 << 7));
                        b = __builtin_bit_cast(uint32_t, m);
                    }
                    o[2 * d + e] = b;
                }
            }
            return __builtin_bit_cast(bf16x8, o);
        } else {
            return __builtin_bit_cast(bf16x8, w);
        }
    }

    template <bool X>
    __device__ __forceinline__ void load_scales(int g) {
        if constexpr (Q) {
            const size_t G = a.K / LTX_GROUP;
#pragma unroll
            for (int j = 0; j < 4; j++) {
                if constexpr (BK == LTX_B_I8_F16S)
                    s[j] = f16_bits_to_f32(((const uint16_t*)sc)[16 * j * G + g]);
                else
                    s[j] = ((const float*)sc)[16 * j * G + g];
                if (X) s[j] *= 16384.0f;
            }
        }
    }

    __device__ __forceinline__ void fold(int i, int j) {
#pragma unroll
        for (int e = 0; e < 4; e++) acc[i][j][e] = __builtin_fmaf(s[j], P[i][j][e], acc[i][j][e]);
    }

    // MFMA m (0 .. 47) of a step: plane m / 16, block m % 16. FIRST: the
    // group's first step, which folds the group before and starts from zero.
    template <bool FIRST, bool FOLD>
    __device__ __forceinline__ void mfma1(int m, const u32x4 (&xa)[12], const bf16x8 (&xb)[4]) {
        const int i = (m >> 2) & 3, j = m & 3;
        const bf16x8 va = __builtin_bit_cast(bf16x8, xa[4 * (m >> 4) + i]);
        if constexpr (Q) {
            if (FOLD && m < 16) fold(i, j);
            P[i][j] = Op<__bf16>::mfma16(va, xb[j], FIRST && m < 16 ? f32x4{0, 0, 0, 0} : P[i][j]);
        } else {
            acc[i][j] = Op<__bf16>::mfma16(va, xb[j], acc[i][j]);
        }
    }

    // One step's 48 MFMAs (xa, xb), with the 16 fragment reads of step STEP of
    // stage RS (W first), the conversion of its W fragments, and, when DMA,
    // the DMA of tile kd into stage DS.
    template <int RS, int STEP, int DS, bool DMA, bool FIRST, bool X>
    __device__ __forceinline__ void region(const u32x4 (&xa)[12], const bf16x8 (&xb)[4], u32x4 (&ya)[12],
                                           bf16x8 (&yb)[4], int kd) {
        WF yw[4];
#pragma unroll
        for (int m = 0; m < 48; m++) {
            mfma1<FIRST, FIRST>(m, xa, xb);
            if (m % 3 == 2) {
                const int g = m / 3;
                __builtin_amdgcn_sched_barrier(0);
                if (g < 4)
                    yw[g] = read_w<RS, STEP>(g);
                else
                    ya[g - 4] = read_a<RS, STEP>(g - 4);
                if (DMA && g < 12 + NDB) dma1<DS>(g, kd);
                __builtin_amdgcn_sched_barrier(0);
            }
            if (m >= 24 && (m - 24) % 6 == 0) yb[(m - 24) / 6] = operand<X>(yw[(m - 24) / 6]);
        }
    }

    // every wave's DMA and LDS reads done
    __device__ __forceinline__ void meet() {
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_waitcnt(7 << 4);  // vmcnt(0) lgkmcnt(0)
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
    }

    // Entered after a barrier: tile k in stage S (k % 2) with its step-1
    // fragments in fa1/fb1, tile k + 1 landed in the other stage, no DMA
    // pending, stage S read by every wave. A group is tiles k, k + 1 of an even k.
    template <int S, bool DMA, bool X>
    __device__ __forceinline__ void pair(int k) {
        if (S == 0) load_scales<X>(k >> 1);
        region<S ^ 1, 0, S, DMA, false, X>(fa1, fb1, fa0, fb0, k + 2);
        __builtin_amdgcn_sched_barrier(0);
        region<S ^ 1, 1, S, false, S == 1, X>(fa0, fb0, fa1, fb1, 0);
        meet();
    }

    // acc = A . W^T of the tile over nk K-tiles (the stages free on entry; the
    // last tile's reads are not waited for)
    template <bool X>
    __device__ __forceinline__ void product(int nk) {
#pragma unroll
        for (int i = 0; i < 4; i++)
#pragma unroll
            for (int j = 0; j < 4; j++) acc[i][j] = f32x4{0, 0, 0, 0};
        dma<0>(0);
        __builtin_amdgcn_s_waitcnt(Q8_WAIT_VM(0));
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
        dma<1>(1);
        {
            WF w0[4], w1[4];
#pragma unroll
            for (int j = 0; j < 4; j++) w0[j] = read_w<0, 0>(j), w1[j] = read_w<0, 1>(j);
#pragma unroll
            for (int i = 0; i < 12; i++) fa0[i] = read_a<0, 0>(i), fa1[i] = read_a<0, 1>(i);
#pragma unroll
            for (int j = 0; j < 4; j++) fb0[j] = operand<X>(w0[j]), fb1[j] = operand<X>(w1[j]);
        }
#pragma unroll
        for (int m = 0; m < 48; m++) mfma1<true, false>(m, fa0, fb0);  // tile 0, step 0
        meet();
        for (int k = 0; k < nk - 2; k += 2) {
            pair<0, true, X>(k);
            pair<1, true, X>(k + 1);
        }
        pair<0, false, X>(nk - 2);
#pragma unroll
        for (int m = 0; m < 48; m++) mfma1<false, false>(m, fa1, fb1);  // tile nk - 1, step 1
        if constexpr (Q)
#pragma unroll
            for (int i = 0; i < 4; i++)
#pragma unroll
                for (int j = 0; j < 4; j++) fold(i, j);
    }

    __device__ __forceinline__ void run(const LtxGemmF3Args& args) {
        const int tid = threadIdx.x, lane = tid & 63;
        const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
        const int wm = 64 * (w >> 1), wn = 64 * (w & 1);
        const int ks_n = a.ksplit > 1 ? a.ksplit : 1;
        const int kc = a.K / ks_n;  // a multiple of 128: nk is even and at least 2
        const int nk = kc / 64;
        const void* planes[3] = {a.a, args.a1, args.a2};
#pragma unroll
        for (int p = 0; p < 3; p++)
            ra_[p] = __builtin_amdgcn_make_buffer_rsrc((void*)planes[p], 0, (int)((uint32_t)a.M * (uint32_t)a.K * 2u),
                                                       Q8_RSRC_W3);
        rb_ = __builtin_amdgcn_make_buffer_rsrc((void*)a.b, 0, (int)((uint32_t)a.N * (uint32_t)a.K * (Q ? 1u : 2u)),
                                                Q8_RSRC_W3);
        wx = a.qxor ^ 0x80808080u;
        // DMA destinations: wave w fills rows 32 w .. 32 w + 31 of each A plane
        // and of W
        la = 4096 * w;
        lb = WOFF + (Q ? 2048 : 4096) * w;
        {
            const int h = lane >> 4, r = lane & 15;
#pragma unroll
            for (int st = 0; st < 2; st++) {
                offa[st] = (wm + r) * 128 + 16 * ((4 * st + h) ^ ((r >> 1) & 7));
                offb[st] = WOFF + (Q ? (wn + r) * 64 + 16 * ((2 * st + (h >> 1)) ^ ((r >> 2) & 3)) + 8 * (h & 1)
                                     : (wn + r) * 128 + 16 * ((4 * st + h) ^ ((r >> 1) & 7)));
            }
        }
        // epilogue patches (32 rows of 72 floats, 9 KB): two waves in each stage
        uint8_t* patch = (w & 1 ? f3_stage<Q, 1>() : f3_stage<Q, 0>()) + 16384 * (w >> 1);
        const int nitems = a.tiles_m * a.tiles_n * ks_n;
        if (Q && tid == 0) f3_redo = 0;  // (before the first tile's barriers)
        for (int item = blockIdx.x; item < nitems; item += gridDim.x) {
            const int ks = item % ks_n;
            const TileIdx ti = tile_of(item / ks_n, a.tiles_m, a.tiles_n);
            const int m0 = ti.tm * 128, n0 = ti.tn * 128;
            const uint32_t k0 = (uint32_t)(ks * kc);  // first k of this slice
            // A and bf16 W: instruction i of wave w fills rows 8 (4 w + i) ..
            // + 7, 8 lanes a row; A rows past M repeat row M - 1
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int tr = 8 * (4 * w + i) + (lane >> 3);
                const int c = (lane & 7) ^ ((tr >> 1) & 7);
                ga[i] = ((uint32_t)min(m0 + tr, a.M - 1) * (uint32_t)a.K + k0) * 2u + 16u * c;
                if constexpr (!Q) gb[i] = ((uint32_t)(n0 + tr) * (uint32_t)a.K + k0) * 2u + 16u * c;
            }
            if constexpr (Q) {
                // int8 W: instruction i of wave w fills rows 16 (2 w + i) .. + 15, 4 lanes a row
                const int nr = lane >> 2, nc = (lane & 3) ^ ((lane >> 4) & 3);
#pragma unroll
                for (int i = 0; i < 2; i++)
                    gb[i] = (uint32_t)(n0 + 16 * (2 * w + i) + nr) * (uint32_t)a.K + k0 + 16u * nc;
                const size_t so = (size_t)(n0 + wn + (lane & 15)) * (a.K / LTX_GROUP) + k0 / LTX_GROUP;
                sc = (const char*)a.scales + so * (BK == LTX_B_I8_F16S ? 2 : 4);
            }
            product<false>(nk);
            if constexpr (Q) {
                float mx = 0.f;  // NaN wins over everything
#pragma unroll
                for (int i = 0; i < 4; i++)
#pragma unroll
                    for (int j = 0; j < 4; j++)
#pragma unroll
                        for (int e = 0; e < 4; e++)
                            mx = __builtin_elementwise_maximum(mx, __builtin_fabsf(acc[i][j][e]));
                if (!(mx <= 3.402823466e38f)) f3_redo = item + 1;
                // (the barrier alone does not keep the compiler from answering the
                // read below with this wave's own store)
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
            }
            meet();
            if constexpr (Q) {
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
                if (__builtin_amdgcn_readfirstlane(f3_redo) == item + 1) {  // the same in every wave
                    product<true>(nk);
                    meet();
                }
            }
            // every wave has passed the last barrier: the stages are free
            const int el = opaque_tid() & 63;
            auto fill = [&](int b, float* p, int LD) {
#pragma unroll
                for (int e = 0; e < 2; e++)
#pragma unroll
                    for (int j = 0; j < 4; j++)
#pragma unroll
                        for (int r = 0; r < 4; r++)
                            p[(16 * e + 4 * (el >> 4) + r) * LD + 16 * j + (el & 15)] = acc[2 * b + e][j][r];
            };
            if (ks_n > 1)
                gemm_store_partial_patch<2, 2>(fill, (float*)patch, a.part + (size_t)ks * a.M * a.N, a.M, a.N, m0 + wm,
                                               n0 + wn);
            else
                gemm_epilogue_patch<__bf16, EPI, 2, 2, decltype(fill), SF, 1>(a, fill, (float*)patch, m0 + wm, n0 + wn,
                                                                             n0);
            // every patch has been read back before the next tile's DMA
            meet();
        }
    }
};

#define F3_GEMM_KERNEL(NAME, BK_, EPI_, SF_)                                           \
    extern "C" __global__ void __launch_bounds__(256, 1) NAME(const LtxGemmF3Args a) { \
        F3Gemm<BK_, EPI_, SF_> k(a.g);                                                 \
        k.run(a);                                                                      \
    }
