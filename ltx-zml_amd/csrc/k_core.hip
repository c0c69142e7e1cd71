// Kernels of the parts around the blocks (ltx/core_parts.zig) and of the
// distilled scheduler (ltx/scheduler.zig). All f32: patchify and the output tail
// at every token count, the conditioning MLPs up to 32 rows (more on the f32 GEMM,
// k_f32.hip).
#include "ltx_device.h"

// DDPM/PixArt sinusoid of t * 1000, cos half first, divisor HALF = 128
// (ltx/core_parts.zig:36-49): freq[k] = exp(k * (-ln(1e4) / 128)) in f32,
// arg = (t * 1000) * freq, out = [cos(arg) | sin(arg)].
__device__ __forceinline__ void core_sinusoid(float t, int k, float& c, float& s) {
    const float freq = expf((float)k * (-9.210340371976184f / 128.0f));
    const float arg = (t * 1000.0f) * freq;
    c = cosf(arg);
    s = sinf(arg);
}
extern "C" __global__ void __launch_bounds__(128) ltx_core_sinusoid(const LtxSinArgs a) {
    const int r = blockIdx.x, k = threadIdx.x;
    if (r >= a.rows) return;
    float c, s;
    core_sinusoid(a.t[r], k, c, s);
    a.out[(size_t)r * 256 + k] = c;
    a.out[(size_t)r * 256 + 128 + k] = s;
}

// y = x * sigmoid(x) (ltx/core_parts.zig:22-24), elementwise.
extern "C" __global__ void __launch_bounds__(256) ltx_core_silu(const LtxEltArgs a) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= a.n) return;
    const float x = a.x[i];
    a.y[i] = x * (1.0f / (1.0f + expf(-x)));
}

// Linear layers of up to R rows in f32 on the VALU: y[r][n] = a[r] . w[n] +
// bias[n], w bf16. Bound by the weights' bytes: a weight is read once, for all
// rows, 16 bytes a lane. A wave takes two consecutive columns n at a time and
// all of K = 4,096 (eight chunks of 512, 8 weights a lane and column); each
// chunk's registers are refilled for the wave's next columns as soon as they
// are used, so 16 KB a wave are in flight. The rows lie in LDS, the 8 values of
// a lane as two float4 512 floats' half apart (a lane stride of 16 B: no bank
// conflicts). The grid is persistent and runs two layers of the same K: the
// timestep branch (job 0, up to R rows) and the prompt branch (job 1, one
// row). Two workgroups a CU up to 4 rows (128 registers a lane): the out
// layers at 3 rows, 369 MB of weights, take 70 us = 5.3 TB/s; with three waves
// a SIMD and the LDS reads lifted out of the loop, the conditioning took 162
// instead of 94 us.
template <int R>
struct RowsDot {
    // acc[r][c] += the chunk's products of rows r and columns c
    static __device__ __forceinline__ void fma8(const float* sa, const u32x4 (&w)[2], float (&acc)[R][2]) {
        float wf[2][8];
#pragma unroll
        for (int c = 0; c < 2; c++)
#pragma unroll
            for (int e = 0; e < 4; e++) {
                wf[c][2 * e] = __builtin_bit_cast(float, w[c][e] << 16);
                wf[c][2 * e + 1] = __builtin_bit_cast(float, w[c][e] & 0xffff0000u);
            }
#pragma unroll
        for (int r = 0; r < R; r++) {
            const f32x4 a0 = *(const f32x4*)(sa + r * LTX_D), a1 = *(const f32x4*)(sa + r * LTX_D + 256);
#pragma unroll
            for (int c = 0; c < 2; c++)
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    acc[r][c] = __builtin_fmaf(a0[e], wf[c][e], acc[r][c]);
                    acc[r][c] = __builtin_fmaf(a1[e], wf[c][4 + e], acc[r][c]);
                }
        }
    }
};

// the layer's outputs from the finished dot product of row r, column n
__device__ __forceinline__ void rows_store(const LtxRowsJob& j, int r, int n, float v) {
    if (r >= j.rows || n >= j.N) return;
    v += j.bias[n];
    const size_t o = (size_t)r * j.N + n;
    if (j.out) j.out[o] = v;
    if (j.act) j.act[o] = v * (1.0f / (1.0f + expf(-v)));
}

template <int R>
__device__ __forceinline__ void rows_job(const LtxRowsJob& j, const float* sa, int g, int step) {
    const int lane = threadIdx.x & 63, ng = j.N / 2;
    if (g >= ng) return;
    const uint16_t* w = j.w + 8 * lane;
    u32x4 buf[8][2];
#pragma unroll
    for (int k = 0; k < 8; k++)
#pragma unroll
        for (int c = 0; c < 2; c++) buf[k][c] = *(const u32x4*)(w + (size_t)(2 * g + c) * LTX_D + 512 * k);
    for (; g < ng; g += step) {
        const int gn = min(g + step, ng - 1);  // past the end: the last columns again
        // the lane's place in the rows, opaque: or the compiler lifts the LDS
        // reads of all chunks out of this loop and spills them (288 B a lane
        // at 3 rows, 1,780 B at 8)
        int lo = 4 * lane;
        asm volatile("" : "+v"(lo));
        float acc[R][2];
#pragma unroll
        for (int r = 0; r < R; r++) acc[r][0] = acc[r][1] = 0.f;
#pragma unroll
        for (int k = 0; k < 8; k++) {
            RowsDot<R>::fma8(sa + 512 * k + lo, buf[k], acc);
#pragma unroll
            for (int c = 0; c < 2; c++) buf[k][c] = *(const u32x4*)(w + (size_t)(2 * gn + c) * LTX_D + 512 * k);
        }
        float mine = 0.f;
#pragma unroll
        for (int r = 0; r < R; r++)
#pragma unroll
            for (int c = 0; c < 2; c++) {
                float v = acc[r][c];
                for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
                if (lane == 2 * r + c) mine = v;
            }
        if (lane < 2 * R) rows_store(j, lane >> 1, 2 * g + (lane & 1), mine);
    }
}

template <int R>
__device__ __forceinline__ void rows_body(const LtxRowsArgs& a) {
    __shared__ __attribute__((aligned(16))) float sa[(R + 1) * LTX_D];
    const int tid = threadIdx.x;
    for (int i = tid; i < (R + 1) * (LTX_D / 4); i += 512) {
        const int r = i / (LTX_D / 4), q = i % (LTX_D / 4);  // float4 q of row r
        const LtxRowsJob& j = a.j[r == R];
        const int rr = r == R ? 0 : r;
        const f32x4 v = rr < j.rows ? *(const f32x4*)(j.a + (size_t)rr * LTX_D + 4 * q) : f32x4{0.f, 0.f, 0.f, 0.f};
        *(f32x4*)(sa + r * LTX_D + (q >> 7) * 512 + (q & 1) * 256 + ((q >> 1) & 63) * 4) = v;
    }
    __syncthreads();
    // columns pairs of job 0, then of job 1, dealt to the grid's waves in turn
    const int nw = gridDim.x * 8, g0 = a.j[0].N / 2;
    int g = blockIdx.x * 8 + (tid >> 6);
    rows_job<R>(a.j[0], sa, g, nw);
    if (g < g0) g += (g0 - g + nw - 1) / nw * nw;
    rows_job<1>(a.j[1], sa + R * LTX_D, g - g0, nw);
}

// The first layers (K = 256) on the sinusoid of t * 1000, which each workgroup
// forms for itself (as ltx_core_sinusoid). A half-wave takes one column.
template <int R>
__device__ __forceinline__ void rows_sin_body(const LtxRowsArgs& a) {
    __shared__ __attribute__((aligned(16))) float sa[(R + 1) * 256];
    const int tid = threadIdx.x;
    for (int i = tid; i < (R + 1) * 128; i += 512) {
        const int r = i >> 7, k = i & 127;
        const LtxRowsJob& j = a.j[r == R];
        const int rr = r == R ? 0 : r;
        float c = 0.f, s = 0.f;
        if (rr < j.rows) core_sinusoid(j.a[rr], k, c, s);
        sa[r * 256 + k] = c;
        sa[r * 256 + 128 + k] = s;
    }
    __syncthreads();
    const int l = tid & 31, n0 = a.j[0].N, nt = n0 + a.j[1].N;
    for (int n = (blockIdx.x * 512 + tid) >> 5; n < nt; n += gridDim.x * 16) {
        const bool one = n >= n0;  // job 1: its single row
        const LtxRowsJob& j = a.j[one];
        const int nn = one ? n - n0 : n;
        const u32x4 w = *(const u32x4*)(j.w + (size_t)nn * 256 + 8 * l);
        float wf[8];
#pragma unroll
        for (int e = 0; e < 4; e++) {
            wf[2 * e] = __builtin_bit_cast(float, w[e] << 16);
            wf[2 * e + 1] = __builtin_bit_cast(float, w[e] & 0xffff0000u);
        }
        const int nr = one ? 1 : R;
        for (int r = 0; r < nr; r++) {
            const float* p = sa + (one ? R : r) * 256 + 8 * l;
            float v = 0.f;
#pragma unroll
            for (int e = 0; e < 8; e++) v = __builtin_fmaf(p[e], wf[e], v);
            for (int o = 16; o > 0; o >>= 1) v += __shfl_xor(v, o, 32);
            if (l == 0) rows_store(j, r, nn, v);
        }
    }
}

#define CORE_ROWS_KERNEL(R)                                                                                            \
    extern "C" __global__ void __launch_bounds__(512, R <= 4 ? 4 : 2) ltx_core_rows_##R(const LtxRowsArgs a) {        \
        rows_body<R>(a);                                                                                              \
    }                                                                                                                  \
    extern "C" __global__ void __launch_bounds__(512) ltx_core_rows_sin_##R(const LtxRowsArgs a) { rows_sin_body<R>(a); }
CORE_ROWS_KERNEL(1)
CORE_ROWS_KERNEL(2)
CORE_ROWS_KERNEL(3)
CORE_ROWS_KERNEL(4)
CORE_ROWS_KERNEL(6)
CORE_ROWS_KERNEL(8)

// Output tail (ltx/core_parts.zig:26-35, 143-166): mean-subtracting LayerNorm
// without weight, biased variance, eps 1e-6, then n * (1 + (fsst[1] + e)) +
// (fsst[0] + e) with e = emb[tidx[t]], times w^T [4096 -> 128] + bias.
// Bound by reading x. A workgroup of 8 waves takes 32 tokens: their statistics
// first, four whole rows a wave; then 256 channels of all of them a step, 32 a
// wave (x a second time, out of the last-level cache: the 32 rows in registers
// would fill them all), normalised, split into three bf16 planes (exact) and
// multiplied with w on bf16 MFMAs, two steps' w and x in flight; the waves'
// partial sums are added in LDS, 16 tokens at a time.
// The modulation rows of a tile whose tokens share one timestep row (all but
// the tiles where the mask changes) are formed once, in LDS. (With the norm a
// launch of its own and the product on the f32 GEMM's T / 128 workgroups, 7,920
// tokens took 57 + 288 us; now 84.)
__shared__ __attribute__((aligned(16))) float tail_mod[2 * LTX_D];  // 1 + scale, shift
__shared__ __attribute__((aligned(16))) float tail_part[8][16][LTX_IN_CH + 4];
__shared__ float tail_mean[32], tail_rstd[32];

template <bool ONE>  // one timestep row in the tile
__device__ __forceinline__ void tail_product(const LtxTailArgs& a, int t0, f32x4 (&acc)[2][8]) {
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int lr = lane & 15, lg = lane >> 4;
    const int c0 = 32 * w + 8 * lg;  // the lane's channels: c0 + 256 ks + 0 .. 7
    const float* x[2];
    const float* e[2];
    float mean[2], r[2];
#pragma unroll
    for (int tb = 0; tb < 2; tb++) {
        const int t = min(t0 + 16 * tb + lr, a.T - 1);
        x[tb] = a.x + (size_t)t * LTX_D + c0;
        e[tb] = a.emb + (size_t)a.tidx[t] * LTX_D + c0;
        mean[tb] = tail_mean[16 * tb + lr];
        r[tb] = tail_rstd[16 * tb + lr];
    }
    const uint16_t* pw = a.w + (size_t)lr * LTX_D + c0;  // row 16 nb + lr of w
    // two steps of x and w in flight: a step's x is reloaded as soon as its
    // planes are formed, its w after its MFMAs
    u32x4 wf[2][8];
    f32x4 xr[2][2][2];
    auto load_w = [&](int b, int ks) {
#pragma unroll
        for (int nb = 0; nb < 8; nb++) wf[b][nb] = *(const u32x4*)(pw + (size_t)16 * nb * LTX_D + 256 * ks);
    };
    auto load_x = [&](int b, int ks) {
#pragma unroll
        for (int tb = 0; tb < 2; tb++)
#pragma unroll
            for (int h = 0; h < 2; h++) xr[b][tb][h] = *(const f32x4*)(x[tb] + 256 * ks + 4 * h);
    };
    auto step = [&](int b, int ks) {
        u32x4 p[2][3];
        f32x4 m1[2], m0[2];
        if (ONE)
#pragma unroll
            for (int h = 0; h < 2; h++) {
                m1[h] = *(const f32x4*)(tail_mod + c0 + 256 * ks + 4 * h);
                m0[h] = *(const f32x4*)(tail_mod + LTX_D + c0 + 256 * ks + 4 * h);
            }
#pragma unroll
        for (int tb = 0; tb < 2; tb++) {
            float y[8];
#pragma unroll
            for (int h = 0; h < 2; h++) {
                if (!ONE) {
                    const f32x4 ev = *(const f32x4*)(e[tb] + 256 * ks + 4 * h);
                    m1[h] = 1.0f + (*(const f32x4*)(a.fsst + LTX_D + c0 + 256 * ks + 4 * h) + ev);
                    m0[h] = *(const f32x4*)(a.fsst + c0 + 256 * ks + 4 * h) + ev;
                }
#pragma unroll
                for (int i = 0; i < 4; i++) y[4 * h + i] = (xr[b][tb][h][i] - mean[tb]) * r[tb] * m1[h][i] + m0[h][i];
            }
            split3(y, p[tb]);
        }
        __builtin_amdgcn_sched_barrier(0);
        load_x(b, min(ks + 2, 15));
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int q = 0; q < 3; q++)
#pragma unroll
            for (int tb = 0; tb < 2; tb++)
#pragma unroll
                for (int nb = 0; nb < 8; nb++)
                    acc[tb][nb] = Op<__bf16>::mfma16(__builtin_bit_cast(bf16x8, p[tb][q]),
                                                     __builtin_bit_cast(bf16x8, wf[b][nb]), acc[tb][nb]);
        __builtin_amdgcn_sched_barrier(0);
        load_w(b, min(ks + 2, 15));
        __builtin_amdgcn_sched_barrier(0);
    };
    load_x(0, 0);
    load_w(0, 0);
    load_x(1, 1);
    load_w(1, 1);
    for (int ks = 0; ks < 16; ks += 2) {
        step(0, ks);
        step(1, ks + 1);
    }
}

extern "C" __global__ void __launch_bounds__(512, 2) ltx_core_tail(const LtxTailArgs a) {
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int lr = lane & 15, lg = lane >> 4;
    const int t0 = blockIdx.x * 32;
    // statistics of rows 4 w .. 4 w + 3, two at a time
#pragma unroll
    for (int g = 0; g < 2; g++) {
        f32x4 v[2][16];
#pragma unroll
        for (int k = 0; k < 2; k++) {
            const float* x = a.x + (size_t)min(t0 + 4 * w + 2 * g + k, a.T - 1) * LTX_D + 4 * lane;
#pragma unroll
            for (int i = 0; i < 16; i++) v[k][i] = *(const f32x4*)(x + 256 * i);
        }
#pragma unroll
        for (int k = 0; k < 2; k++) {
            auto sum = [](f32x4 s4) {
                float s = (s4[0] + s4[1]) + (s4[2] + s4[3]);
                for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
                return s;
            };
            f32x4 s4 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int i = 0; i < 16; i++) s4 += v[k][i];
            const float mean = sum(s4) / (float)LTX_D;
            s4 = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int i = 0; i < 16; i++) {
                const f32x4 d = v[k][i] - mean;
                s4 += d * d;
            }
            const float var = sum(s4) / (float)LTX_D;
            if (lane == 0) {
                tail_mean[4 * w + 2 * g + k] = mean;
                tail_rstd[4 * w + 2 * g + k] = 1.0f / sqrtf(var + 1e-6f);
            }
        }
    }
    const int k0 = a.tidx[t0];
    const bool one = __builtin_amdgcn_ballot_w64(a.tidx[min(t0 + (lane & 31), a.T - 1)] != k0) == 0;  // the same in every wave
    if (one) {
        const float* e = a.emb + (size_t)k0 * LTX_D;
        for (int c = 4 * tid; c < LTX_D; c += 2048) {
            const f32x4 ev = *(const f32x4*)(e + c);
            *(f32x4*)(tail_mod + c) = 1.0f + (*(const f32x4*)(a.fsst + LTX_D + c) + ev);
            *(f32x4*)(tail_mod + LTX_D + c) = *(const f32x4*)(a.fsst + c) + ev;
        }
    }
    __syncthreads();
    f32x4 acc[2][8];
#pragma unroll
    for (int tb = 0; tb < 2; tb++)
#pragma unroll
        for (int nb = 0; nb < 8; nb++) acc[tb][nb] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (one)
        tail_product<true>(a, t0, acc);
    else
        tail_product<false>(a, t0, acc);
    // acc[tb][nb][i]: token 16 tb + 4 lg + i, column 16 nb + lr
    const int row = tid >> 5, c = 4 * (tid & 31);
#pragma unroll
    for (int tb = 0; tb < 2; tb++) {
        if (tb) __syncthreads();
#pragma unroll
        for (int nb = 0; nb < 8; nb++)
#pragma unroll
            for (int i = 0; i < 4; i++) tail_part[w][4 * lg + i][16 * nb + lr] = acc[tb][nb][i];
        __syncthreads();
        f32x4 o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < 8; i++) o += *(const f32x4*)&tail_part[i][row][c];
        const int t = t0 + 16 * tb + row;
        if (t < a.T) {
            float* dst = a.vel + (size_t)t * LTX_IN_CH + c;  // (of any 4-byte alignment)
#pragma unroll
            for (int i = 0; i < 4; i++) dst[i] = o[i] + a.bias[c + i];
        }
    }
}

// Patchify (ltx/core_parts.zig:112-121): x = lat . w^T + bias, 128 -> 4096.
// Bound by writing x. A workgroup of 8 waves takes 64 tokens and 512 columns:
// the latents go to LDS once as three bf16 planes (exact), each wave holds the
// weights of its 64 columns in registers, and the loop over the token blocks
// then reads LDS only. (With weights loaded in a loop over the columns, each
// load's wait also waited for the stores before it: 59 us against 41 at 7,920
// tokens; on the f32 GEMM 95.) w's rows are the MFMA's A operand, so a lane's results are four
// consecutive columns of one token.
// LDS rows of 256 B a token and plane, 16-byte chunk c of token t in slot
// c ^ (t & 15): the 16 tokens of a fragment read cover all banks.
extern "C" __global__ void __launch_bounds__(512, 4) ltx_core_patchify(const LtxPatchifyArgs a) {
    __shared__ __attribute__((aligned(16))) uint8_t planes[3][64 * 256];
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int lr = lane & 15, lg = lane >> 4;
    const int t0 = blockIdx.x * 64, n0 = 512 * blockIdx.y + 64 * w;
    u32x4 wf[4][4];  // [16 columns][32 channels]
#pragma unroll
    for (int nb = 0; nb < 4; nb++)
#pragma unroll
        for (int ks = 0; ks < 4; ks++)
            wf[nb][ks] = *(const u32x4*)(a.w + (size_t)(n0 + 16 * nb + lr) * LTX_IN_CH + 32 * ks + 8 * lg);
#pragma unroll
    for (int i = 0; i < 2; i++) {
        const int id = tid + 512 * i, t = id >> 4, c = id & 15;  // chunk c (8 channels) of token t0 + t
        const float* l = a.lat + (size_t)min(t0 + t, a.T - 1) * LTX_IN_CH + 8 * c;
        const f32x4 l0 = *(const f32x4*)l, l1 = *(const f32x4*)(l + 4);
        u32x4 p[3];
        split3({l0[0], l0[1], l0[2], l0[3], l1[0], l1[1], l1[2], l1[3]}, p);
#pragma unroll
        for (int q = 0; q < 3; q++) *(u32x4*)(planes[q] + 256 * t + 16 * (c ^ (t & 15))) = p[q];
    }
    f32x4 b[4];
#pragma unroll
    for (int nb = 0; nb < 4; nb++) b[nb] = *(const f32x4*)(a.bias + n0 + 16 * nb + 4 * lg);
    __syncthreads();
#pragma unroll
    for (int tb = 0; tb < 4; tb++) {
        f32x4 acc[4];
#pragma unroll
        for (int nb = 0; nb < 4; nb++) acc[nb] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int q = 0; q < 3; q++)
#pragma unroll
            for (int ks = 0; ks < 4; ks++) {
                const u32x4 f = *(const u32x4*)(planes[q] + 256 * (16 * tb + lr) + 16 * ((4 * ks + lg) ^ lr));
#pragma unroll
                for (int nb = 0; nb < 4; nb++)
                    acc[nb] = Op<__bf16>::mfma16(__builtin_bit_cast(bf16x8, wf[nb][ks]), __builtin_bit_cast(bf16x8, f),
                                                 acc[nb]);
            }
        const int t = t0 + 16 * tb + lr;
        if (t < a.T)
#pragma unroll
            for (int nb = 0; nb < 4; nb++) *(f32x4*)(a.x + (size_t)t * LTX_D + n0 + 16 * nb + 4 * lg) = acc[nb] + b[nb];
    }
}

// One Euler step of the distilled sampler on the latent [T][C], in the
// reference's exact f32 operation order and without fused multiply-adds
// (ltx/scheduler.zig:54-80):
//   den  = x - v * ts                       (toDenoised, per-token ts)
//   post = den * m + c * (1 - m)            (postProcess)
//   next = x + ((x - post) / sigma) * dt    (eulerStep, dt = sigma_next - sigma)
// with ts = tk[tidx[t]], m = maskk[tidx[t]] for token t.
extern "C" __global__ void __launch_bounds__(256) ltx_sched_step(const LtxSchedArgs a) {
#pragma clang fp contract(off)
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= a.n) return;
    const int k = a.tidx[i / a.stride];
    const float ts = a.tk[k], m = a.maskk[k];
    const float x = a.x[i];
    const float vts = a.v[i] * ts;
    const float den = x - vts;
    const float dm = den * m;
    const float om = 1.0f - m;
    const float cm = a.clean[i] * om;
    const float post = dm + cm;
    const float dt = a.sigma_next - a.sigma;
    const float vel = (x - post) / a.sigma;
    const float step = vel * dt;
    a.y[i] = x + step;
}

// torch.lerp as the reference computes it (ltx/scheduler.zig:21-33): the
// branch on |w| < 0.5 and one fused multiply-add in either branch.
__device__ __forceinline__ float sched_lerp(float a, float b, float w) {
#pragma clang fp contract(off)
    const float d = b - a;
    if (fabsf(w) < 0.5f) return __builtin_fmaf(w, d, a);
    return __builtin_fmaf(-d, 1.0f - w, b);
}

// GaussianNoiser at state initialisation (ltx/scheduler.zig:38-46):
// x = lerp(clean, noise, noise_scale); out = lerp(clean, x, mask[token]).
extern "C" __global__ void __launch_bounds__(256) ltx_sched_noise_init(const LtxNoiseArgs a) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= a.n) return;
    const float c = a.clean[i];
    const float x = sched_lerp(c, a.noise[i], a.noise_scale);
    a.y[i] = sched_lerp(c, x, a.maskk[a.tidx[i / a.stride]]);
}

// t[k] = mask[k] * sigma (ltx/scheduler.zig:48-51), one value per distinct
// mask value, and t[K] = sigma itself (the prompt conditioning's input), so a
// step needs no host-to-device copy. K < 64.
extern "C" __global__ void __launch_bounds__(64) ltx_sched_timesteps(const LtxTimestepArgs a) {
#pragma clang fp contract(off)
    const int k = threadIdx.x;
    if (k < a.K) a.tk[k] = a.maskk[k] * a.sigma;
    else if (k == a.K) a.tk[k] = a.sigma;
}
