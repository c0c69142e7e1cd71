// Block forward orchestration: QBlock.qBlockOutAll (ltx/block.zig:544-574)
// as a sequence of gfx950 kernel launches on one stream, plus the isolated
// operator entry points.
#include <cmath>
#include <algorithm>
#include <cstring>
#include <new>
#include <numeric>

#include "ltx_internal.hpp"

namespace ltx {

static const char* msuffix(int mode) { return mode == LTX_MODE_BF16 ? "bf16" : "f16"; }

static size_t al(size_t n) { return (n + 255) & ~(size_t)255; }

// V^T's row stride: the keys in whole 64-key attention tiles.
static int vt_ld(size_t n) { return (int)((n + 63) & ~(size_t)63); }

// Bump allocator over the context workspace.
struct Carve {
    char* base;
    size_t off = 0;
    size_t total = 0;
    bool dry;
    void* take(size_t n) {
        void* p = dry ? nullptr : base + off;
        off += al(n);
        return p;
    }
};

struct Ws16 {
    void *n_msa, *qk16, *vt1, *qh1, *kh1, *glog1, *o1, *x_sa, *attn_in, *q2_16, *glog2, *enc, *k2_16, *vt2, *qh2,
        *kh2, *o2, *x_ca, *ff_in, *h, *part, *part2;
    void *v1, *v2;  // the stages of V: V^T's rows without padding (vt1, vt2 themselves where they have none)
    void* dq[6];  // 16-bit weights of qkv1, o1, q2, o2, ff1, ff2 for the four-wave GEMM (NULL: not used)
};

// The projections the four-wave GEMM may take, as (N, K) with A rows of K
// elements and M = T: qkv1, o1, q2, o2, ff1, ff2.
static const int kX4Shapes[6][2] = {{3 * LTX_D, LTX_D}, {LTX_D, LTX_D}, {LTX_D, LTX_D},
                                    {LTX_D, LTX_D},     {LTX_FF, LTX_D}, {LTX_D, LTX_FF}};

// Split-K slices of a GEMM whose 256 x tn output tiles would fill at most
// half the CUs: the largest power of two S <= 8 with tiles * S <= CUs and
// K / S a multiple of 128 of at least 512 (eight K-tiles per slice).
static int gemm_ksplit(int num_cu, int M, int N, int K, int tn = 256, int tm = 256) {
    const int tiles = ((M + tm - 1) / tm) * (N / tn);
    int s = 1;
    while (s < 8 && tiles * s * 2 <= num_cu && K % (256 * s) == 0 && K / (s * 2) >= 512) s *= 2;
    return s;
}

// Rows of a persistent GEMM's 256-column tiles, 256 or 192: the height whose
// whole rounds of one tile a CU are the fewest rows, a row of the lower tiles
// counted 1.08 times, past K = 4,096 1.2 times (they read more LDS, move more
// operand bytes and dequantise more weights per MFMA).
// Measured, 192 against 256 rows, us (rows x N x K, the dequantisation
// included; rounds of each):
// equal rounds 4,100 x 4,096 x 4,096 151 : 187, 2,970 x 12,288 x 4,096 284 :
// 313, 1,600 x 12,288 x 4,096 170 : 193, 4,100 x 4,096 x 16,384 604 : 683, 9,216
// x 4,096 x 16,384 1,131 : 1,246;
// six to five 5,400 x 12,288 x 4,096 458 : 483, 18,432 x 4,096 x 4,096 462 :
// 470, 17,000 x 4,096 x 16,384 2,176 : 2,009; eleven to nine 16,500 x 8,192 x
// 4,096 834 : 855; five to four 4,100 x 12,288 x 4,096 383 : 390, 15,360 x 4,096
// x 4,096 388 : 384, 3,500 x 16,384 x 4,096 434 : 421, 13,000 x 4,096 x 16,384
// 1,822 : 1,632; fifteen to twelve 15,000 x 12,288 x 4,096 1,165 : 1,156;
// one round of the W8A16 kernel with f32 scales 2,100 x 4,096 x 4,096 82 : 86,
// 2,500 94 : 91, yet in a block, between other kernels, the lower tiles win there
// (bf16, 2,304 tokens 1,308 : 1,356, 2,500 tokens 1,424 : 1,438).
static int tile_rows(const ltx_ctx* c, int M, int N, int K) {
    if (c->gemm_rows == 192 || c->gemm_rows == 256) return c->gemm_rows;
    auto rounds = [&](int rows) { return (((M + rows - 1) / rows) * (N / 256) + c->num_cu - 1) / c->num_cu; };
    return rounds(192) * 192 * (K <= 4096 ? 1.08f : 1.2f) < rounds(256) * 256 ? 192 : 256;
}

bool x4_shape(const ltx_ctx* c, int mode, int M, int N, int K, int lda, bool w16) {
    if (mode != LTX_MODE_F16 && mode != LTX_MODE_BF16) return false;
    if (!c->gemm_x4 || !c->gemm_dma) return false;
    if (M <= 0 || N % 256 || K % 128 || lda < K || lda % 8) return false;
    if ((uint64_t)M * lda * 2 >= (1ull << 31) || (uint64_t)N * K * 2 >= (1ull << 31)) return false;
    if (c->gemm_x4 == 2) return true;
    // where its 256 x 256 tiles fill the CUs: the sizes that need no split-K.
    // 16-bit weights (no dequantisation): as soon as the 256 x 128 tiles of the
    // other kernel need a second round for 4,096 columns (o1 and o2 at 2,970
    // rows 84 against 120 us; the whole unquantised block in bf16, before and
    // with it: 2,049 tokens 1,592 : 1,290 us, 2,500 1,670 : 1,328, 2,970 1,883 :
    // 1,572, 4,000 2,131 : 1,960; 2,048 tokens, on the other kernel, 1,030)
    return M >= (w16 ? 2049 : 4096) && gemm_ksplit(c->num_cu, M, N, K) == 1;
}

bool s4_shape(const ltx_ctx* c, int mode, int M, int N, int K, int lda, bool q8) {
    if (mode != LTX_MODE_F16 && mode != LTX_MODE_BF16) return false;
    if (!c->gemm_s4 || !c->gemm_dma) return false;
    if (M <= 0 || N % 128 || K % 128 || lda < K || lda % 8) return false;
    if ((uint64_t)M * lda * 2 >= (1ull << 31) || (uint64_t)N * K * (q8 ? 1 : 2) >= (1ull << 31)) return false;
    if (c->gemm_s4 == 2) return true;
    // int8 weights where the 256 x 256 kernels would split K (their tiles
    // fill at most half the CUs) over at most 4,096: there it needs no
    // split-K reduce (the context k|v projection, the 4096-wide projections
    // below 4,096 rows). With 16-bit weights, or K = 16,384, its 128 x 128
    // tiles (half the flops per byte moved) measured slower than the split
    // 256 x 256 kernels; with no split (q|k|v at 1,024 rows) slower too. Up to
    // 256 rows it takes K = 16,384 as well, half or all of whose 256-row tiles
    // would be padding: 16 x 4,096 x 16,384 34 against 57 us, 128 rows 37 : 58,
    // 256 rows 55 : 58; 400 rows 90 : 82.
    return q8 && M < 4096 && (K <= 4096 || M <= 256) && gemm_ksplit(c->num_cu, M, N, K) > 1;
}

// Whether the f32 GEMM on bf16 MFMAs takes an M x N x K product (shape and
// 31-bit buffer offsets; gemm32 checks the alignment of the operands). It does
// wherever it can: at 1,024 rows it takes a third of the f32 MFMA kernel's time
// and below that its split-K fills the chip where the other has N / 128
// workgroups a row tile.
bool f3_shape(const ltx_ctx* c, int M, int N, int K) {
    return c->gemm_f3 && M > 0 && N % 128 == 0 && K % 128 == 0 && K <= (1 << 15) && (uint64_t)M * K * 2 < (1ull << 31) &&
           (uint64_t)N * K * 2 < (1ull << 31);
}
// Its scratch: the three planes of A, and the split-K partial sums (0: no split).
size_t f3_planes_bytes(int M, int K) { return 3 * al((size_t)M * K * 2); }
size_t f3_part_bytes(const ltx_ctx* c, int M, int N, int K) {
    const int s = gemm_ksplit(c->num_cu, M, N, K, 128, 128);
    return s > 1 ? (size_t)s * M * N * 4 : 0;
}

int f3_rows(const ltx_ctx* c, int M, int N, int K, size_t room) {
    const size_t row = 3 * (size_t)K * 2 + f3_part_bytes(c, M, N, K) / M, pad = 3 * 256;  // al() of three planes
    if (room < pad) return 0;
    const size_t most = (room - pad) / row;
    if (most >= (size_t)M) return M;
    // whole rounds of one tile a CU, or a pass's last round idles (28,672 x 4,096
    // x 16,384 in six even passes 12.1 ms, in whole rounds and in one pass 11.4)
    const int tiles = (int)(most / 128), q = c->num_cu / std::gcd(N / 128, c->num_cu);
    return (tiles >= q ? tiles / q * q : tiles) * 128;
}

// Whether the small-grid kernel gathers the isolated GEMM's scales as packed
// instead of from the words that a launch of 5 us lays out: the gathers cost more
// with more row tiles on the chip. Measured, packed against words, us (rows x N,
// K = 4,096): 16 x 4,096 17.8 : 21.4, 128 x 4,096 24.2 : 27.4, 256 x 8,192 34.5 :
// 36.3; 300 x 4,096 34.1 : 35.7, x 8,192 43.3 : 42.2, x 16,384 65.3 : 66.4; 448 x
// 8,192 44.8 : 43.6, bf16 x 16,384 85.9 : 84.3; 512 x 8,192 45.4 : 44.6, 1,024 x
// 4,096 49.4 : 45.2.
static bool s4_packed_scales(int M) { return M <= 256; }

// The small-T schedule of the block forward (side stream from the first
// RMSNorm + modulate on).
static bool side_early(const ltx_ctx* c, size_t T) {
    return c->side_early == 2 || (c->side_early == 1 && T < (size_t)kEarlySideRows);
}

static void carve16(Carve& c, Ws16& w, size_t T, size_t S, const ltx_ctx* ctx, int mode) {
    const size_t D = LTX_D;
    const int num_cu = ctx->num_cu;
    w.n_msa = c.take(T * D * 2);
    w.qk16 = c.take(T * 2 * D * 2);
    w.vt1 = c.take((size_t)vt_ld(T) * D * 2);
    w.v1 = (size_t)vt_ld(T) != T ? c.take(T * D * 2) : w.vt1;
    w.qh1 = c.take(T * D * 2);
    w.kh1 = c.take(T * D * 2);
    w.glog1 = c.take(T * LTX_H * 4);
    w.o1 = c.take(T * D * 2);
    w.x_sa = c.take(T * D * 4);
    w.attn_in = c.take(T * D * 2);
    w.q2_16 = c.take(T * D * 2);
    w.glog2 = c.take(T * LTX_H * 4);
    w.enc = c.take(S * D * 2);
    w.k2_16 = c.take(S * D * 2);
    w.vt2 = c.take((size_t)vt_ld(S) * D * 2);
    w.v2 = (size_t)vt_ld(S) != S ? c.take(S * D * 2) : w.vt2;
    w.qh2 = c.take(T * D * 2);
    w.kh2 = c.take(S * D * 2);
    w.o2 = c.take(T * D * 2);
    w.x_ca = c.take(T * D * 4);
    w.ff_in = c.take(T * D * 2);
    w.h = c.take(T * LTX_FF * 2);
    // f32 partial sums of the split-K GEMMs: the largest slices * M * N over
    // the block's seven projections (none at large T)
    size_t part = 0;
    const int shapes[6][3] = {{(int)T, 3 * LTX_D, LTX_D}, {(int)T, LTX_D, LTX_D}, {(int)S, 2 * LTX_D, LTX_D},
                              {(int)T, LTX_FF, LTX_D}, {(int)T, LTX_D, LTX_FF}, {(int)T, LTX_D, LTX_D}};
    for (const auto& sh : shapes) {
        const int k = gemm_ksplit(num_cu, sh[0], sh[1], sh[2]);
        if (k > 1) part = std::max(part, (size_t)k * sh[0] * sh[1] * 4);
    }
    w.part = part ? c.take(part) : nullptr;
    // the context k|v GEMM's own partial sums when it runs on the side
    // stream beside the main chain's split GEMMs
    w.part2 = nullptr;
    if (side_early(ctx, T)) {
        const int k = gemm_ksplit(num_cu, (int)S, 2 * LTX_D, LTX_D);
        if (k > 1) w.part2 = c.take((size_t)k * S * 2 * LTX_D * 4);
    }
    for (int i = 0; i < 6; i++) {
        const int N = kX4Shapes[i][0], K = kX4Shapes[i][1];
        w.dq[i] = x4_shape(ctx, mode, (int)T, N, K, K) ? c.take((size_t)N * K * 2) : nullptr;
    }
}

struct Ws32 {
    void *n_msa, *q, *k, *v, *glog1, *o1, *x_sa, *attn_in, *q2, *enc, *k2, *v2, *glog2, *o2, *x_ca, *ff_in, *h;
    void *planes, *part;  // the f3 GEMMs' split of the current A (three bf16 planes) and split-K partial sums
    size_t planes_bytes;
};

static void carve32(Carve& c, Ws32& w, size_t T, size_t S, const ltx_ctx* ctx) {
    const size_t D = LTX_D;
    w.n_msa = c.take(T * D * 4);
    w.q = c.take(T * D * 4);
    w.k = c.take(T * D * 4);
    w.v = c.take(T * D * 4);
    w.glog1 = c.take(T * LTX_H * 4);
    w.o1 = c.take(T * D * 4);
    w.x_sa = c.take(T * D * 4);
    w.attn_in = c.take(T * D * 4);
    w.q2 = c.take(T * D * 4);
    w.enc = c.take(S * D * 4);
    w.k2 = c.take(S * D * 4);
    w.v2 = c.take(S * D * 4);
    w.glog2 = c.take(T * LTX_H * 4);
    w.o2 = c.take(T * D * 4);
    w.x_ca = c.take(T * D * 4);
    w.ff_in = c.take(T * D * 4);
    w.h = c.take(T * LTX_FF * 4);
    w.planes = w.part = nullptr;
    size_t planes = 0, part = 0;
    const int shapes[4][3] = {{(int)T, LTX_D, LTX_D}, {(int)S, LTX_D, LTX_D}, {(int)T, LTX_FF, LTX_D},
                              {(int)T, LTX_D, LTX_FF}};
    for (const auto& sh : shapes) {
        if (!ctx->ws_planes || !f3_shape(ctx, sh[0], sh[1], sh[2])) continue;
        planes = std::max(planes, f3_planes_bytes(sh[0], sh[2]));
        part = std::max(part, f3_part_bytes(ctx, sh[0], sh[1], sh[2]));
    }
    if (planes) w.planes = c.take(planes);
    w.planes_bytes = planes;
    if (part) w.part = c.take(part);
}

// Room for a forward. Mode F32's planes only where there is room for them too: a
// forward without runs its GEMMs on the f32 MFMA kernel, as before they had any.
// grow: may allocate for them (not in a capture).
static void ensure_ws(ltx_ctx* c, size_t T, size_t S, int mode, bool grow = true) {
    auto need = [&]() {
        Carve cv{nullptr, 0, 0, true};
        if (mode == LTX_MODE_F32) {
            Ws32 w;
            carve32(cv, w, T, S, c);
        } else {
            Ws16 w;
            carve16(cv, w, T, S, c, mode);
        }
        return cv.off;
    };
    c->ws_planes = true;
    size_t n = need();
    if (mode == LTX_MODE_F32 && c->ws.bytes < n) {
        c->ws_planes = false;
        const size_t least = need();
        c->ws_planes = n > least && grow && !c->ws_pins && hipDeviceSynchronize() == hipSuccess && c->ws.try_grow(n);
        if (!c->ws_planes) n = least;
    }
    if (c->ws.bytes < n) {
        if (c->ws_pins)
            throw Error("the workspace is bound by " + std::to_string(c->ws_pins) +
                        " live block graph(s) and this forward needs a larger one; destroy them first");
        HIPC(hipDeviceSynchronize());
        c->ws.alloc(n);
    }
}

// ---- launch helpers -------------------------------------------------------

static LtxAda make_ada(const ltx_block_weights* w, const float* tstab, const int32_t* tidx, int K) {
    LtxAda a;
    a.sst = (const float*)w->sst.p;
    a.tstab = tstab;
    a.tidx = tidx;
    a.K = K;
    return a;
}

// The range guard's counter for the 16-bit modes (NULL in mode F32).
static unsigned long long* sat_of(ltx_ctx* c, int mode) {
    return mode == LTX_MODE_F32 ? nullptr : (unsigned long long*)c->range_ctr.p;
}

// sat_add: a device count the kernel adds to the range guard (the weights'
// f16_over in mode F16), or NULL.
static void norm_mod(ltx_ctx* c, int mode, const float* x, void* y, LtxAda ada, int rows, int ish, int isc,
                     hipStream_t st, const unsigned long long* sat_add = nullptr) {
    LtxNormArgs a{x, y, ada, rows, ish, isc, sat_of(c, mode), sat_add};
    const char* k = mode == LTX_MODE_F32 ? "ltx_norm_mod_f32" : mode == LTX_MODE_BF16 ? "ltx_norm_mod_bf16" : "ltx_norm_mod_f16";
    c->launch(k, (rows + 3) / 4, 1, 1, 256, &a, st);  // four rows per workgroup (NORM_ROWS)
}

// 16-bit GEMM: y = A . W^T with the given epilogue. w16: the int8
// projection's weights dequantised to the operand type for this call (by
// dequant16), which routes it to the four-wave kernel, or NULL.
static void gemm16(ltx_ctx* c, int mode, const LtxProj& p, const void* A, int M, int lda, int epi, LtxGemmArgs g,
                   hipStream_t st, const char* label = nullptr, const void* w16 = nullptr) {
    if (p.N % 256 != 0 || p.K % 64 != 0) throw Error("gemm16: N must be a multiple of 256 and K of 64");
    g.a = A;
    g.M = M;
    g.N = p.N;
    g.K = p.K;
    g.lda = lda;
    g.bias = (const float*)p.bias.p;
    const char* bk;
    if (p.q8) {
        g.b = p.q.p;
        g.scales = p.s.p;
        g.qxor = p.qflip ? 0u : 0x80808080u;
        bk = p.scale_f16 ? "i8f16" : "i8f32";
    } else {
        g.b = mode == LTX_MODE_BF16 ? p.w_bf16.p : p.w_f16.p;
        g.scales = nullptr;
        bk = "w16";
    }
    if (!g.b) throw Error("gemm16: weight not resident for this mode");
    g.tiles_m = (M + 255) / 256;
    g.tiles_n = p.N / 256;
    char name[64];
    auto al16 = [](const void* q) { return ((uintptr_t)q & 15) == 0; };
    const char* es = epi == LTX_EPI_STORE ? "store" : epi == LTX_EPI_RESID_GATE ? "resid" : "qkv";
    // Four-wave 16-bit kernel: unquantised weights, or int8 weights
    // dequantised for this call; 16-byte aligned operands (its DMA and
    // epilogue move 16-byte vectors)
    {
        const void* wb = p.q8 ? w16 : (mode == LTX_MODE_BF16 ? p.w_bf16.p : p.w_f16.p);
        if (wb && x4_shape(c, mode, M, p.N, p.K, lda, !p.q8) && g.ldo % 8 == 0 && al16(A) && al16(wb) && al16(g.out) &&
            al16(g.out2) && al16(g.resid) && al16(g.bias) && al16(g.ada.tstab) && al16(g.ada.sst)) {
            g.b = wb;
            g.scales = nullptr;
            g.ksplit = 1;
            std::snprintf(name, sizeof(name), "ltx_gemm_x4_%s_%s%s%s", msuffix(mode), es,
                          epi == LTX_EPI_STORE && g.out_f32 ? "32" : "", epi == LTX_EPI_STORE && g.gelu ? "_gelu" : "");
            const int tr = tile_rows(c, M, p.N, p.K);
            if (tr != 256) std::snprintf(name + std::strlen(name), sizeof(name) - std::strlen(name), "_h%d", tr);
            g.tiles_m = (M + tr - 1) / tr;
            const int nitems = g.tiles_m * g.tiles_n;
            c->launch(name, c->gemm_persistent ? std::min(nitems, c->num_cu) : nitems, 1, 1, 256, &g, st, label);
            return;
        }
    }
    // Small grids: 128 x 128 tiles, two workgroups a CU, int8 weights laid
    // out for the LDS-DMA kernels (bytes q + 128, scale words) or 16-bit
    // weights; split K only while even those tiles fill at most half the CUs
    {
        const void* wb = p.q8 ? ((p.qraw && s4_packed_scales(M)) || ((p.qflip || p.qraw) && p.s2.p) ? p.q.p : nullptr) : (mode == LTX_MODE_BF16 ? p.w_bf16.p : p.w_f16.p);
        if (wb && s4_shape(c, mode, M, p.N, p.K, lda, p.q8) && g.ldo % 8 == 0 && al16(A) && al16(wb) && al16(g.out) &&
            al16(g.out2) && al16(g.resid) && al16(g.bias) && al16(g.ada.tstab) && al16(g.ada.sst)) {
            g.b = wb;
            const bool sp = p.qraw && s4_packed_scales(M);
            g.scales = !p.q8 ? nullptr : sp ? p.s.p : p.s2.p;
            g.tiles_m = (M + 127) / 128;
            g.tiles_n = p.N / 128;
            g.ksplit = g.part ? gemm_ksplit(c->num_cu, M, p.N, p.K, 128, 128) : 1;
            std::snprintf(name, sizeof(name), "ltx_gemm_s4_%s_%s_%s%s", msuffix(mode),
                          p.q8 ? (p.scale_f16 ? "i8f16" : "i8f32") : "w16", es, sp ? "_packed" : p.qraw ? "_raw" : "");
            const int nitems = g.tiles_m * g.tiles_n * g.ksplit;
            c->launch(name, c->gemm_persistent ? std::min(nitems, 2 * c->num_cu) : nitems, 1, 1, 256, &g, st, label);
            if (g.ksplit > 1) {
                std::snprintf(name, sizeof(name), "ltx_gemm_reduce_%s_%s", msuffix(mode), es);
                c->launch(name, p.N / 64, (M + 63) / 64, 1, 256, &g, st, "splitk_reduce");
            }
            return;
        }
    }
    // LDS-DMA int8 kernel: f16 or bf16 operands, f16 scales, K a multiple of
    // 128, and byte offsets of A and W within 31 bits (32-bit buffer offsets)
    if ((mode == LTX_MODE_F16 || mode == LTX_MODE_BF16) && p.q8 && (p.qflip || p.qraw) && p.s2.p &&
        c->gemm_dma && p.K % 128 == 0 && (uint64_t)M * lda * 2 < (1ull << 31) && (uint64_t)p.N * p.K < (1ull << 31) && g.ldo % 8 == 0 &&
        al16(g.out) && al16(g.out2) && al16(g.resid) && al16(g.bias) && al16(g.ada.tstab) && al16(g.ada.sst)) {
        // (its epilogue moves 16-byte vectors: outputs, residual and bias 16-byte aligned)
        g.scales = p.s2.p;
        std::snprintf(name, sizeof(name), "ltx_gemm_q8_%s%s%s%s", mode == LTX_MODE_BF16 ? "bf16_" : "",
                      p.scale_f16 ? "" : "s32_", es, p.qraw ? "_raw" : "");
        // few output tiles: split K over more workgroups (when the caller
        // gave a buffer for the partial sums), then reduce + epilogue
        g.ksplit = g.part ? gemm_ksplit(c->num_cu, M, p.N, p.K) : 1;
        const int tr = g.ksplit > 1 ? 256 : tile_rows(c, M, p.N, p.K);
        if (tr != 256) std::snprintf(name + std::strlen(name), sizeof(name) - std::strlen(name), "_h%d", tr);
        g.tiles_m = (M + tr - 1) / tr;
        const int nitems = g.tiles_m * g.tiles_n * g.ksplit;
        c->launch(name, c->gemm_persistent ? std::min(nitems, c->num_cu) : nitems, 1, 1, 512, &g, st, label);
        if (g.ksplit > 1) {
            std::snprintf(name, sizeof(name), "ltx_gemm_reduce_%s_%s", msuffix(mode), es);
            c->launch(name, p.N / 64, (M + 63) / 64, 1, 256, &g, st, "splitk_reduce");
        }
        return;
    }
    // LDS-DMA 16-bit-weight kernel (256 x 128 tiles): the same conditions
    if ((mode == LTX_MODE_F16 || mode == LTX_MODE_BF16) && !p.q8 && c->gemm_dma && p.K % 128 == 0 &&
        p.N % 128 == 0 && (uint64_t)M * lda * 2 < (1ull << 31) && (uint64_t)p.N * p.K * 2 < (1ull << 31) &&
        g.ldo % 8 == 0 && al16(g.out) && al16(g.out2) && al16(g.resid) && al16(g.bias) && al16(g.ada.tstab) &&
        al16(g.ada.sst) && al16(g.b)) {
        std::snprintf(name, sizeof(name), "ltx_gemm_w16dma_%s_%s", msuffix(mode), es);
        g.tiles_n = p.N / 128;
        g.ksplit = g.part ? gemm_ksplit(c->num_cu, M, p.N, p.K, 128) : 1;
        const int nitems = g.tiles_m * g.tiles_n * g.ksplit;
        c->launch(name, c->gemm_persistent ? std::min(nitems, c->num_cu) : nitems, 1, 1, 512, &g, st, label);
        if (g.ksplit > 1) {
            std::snprintf(name, sizeof(name), "ltx_gemm_reduce_%s_%s", msuffix(mode), es);
            c->launch(name, p.N / 64, (M + 63) / 64, 1, 256, &g, st, "splitk_reduce");
        }
        return;
    }
    std::snprintf(name, sizeof(name), "ltx_gemm_%s_%s_%s", msuffix(mode), bk, es);
    // split-K as above; the reduce kernel moves 16-byte vectors, so only with
    // aligned operands
    const bool aligned = g.ldo % 8 == 0 && al16(g.out) && al16(g.out2) && al16(g.resid) && al16(g.bias) &&
                         al16(g.ada.tstab) && al16(g.ada.sst);
    g.ksplit = g.part && aligned ? gemm_ksplit(c->num_cu, M, p.N, p.K) : 1;
    c->launch(name, g.tiles_m * g.tiles_n * g.ksplit, 1, 1, 512, &g, st, label);
    if (g.ksplit > 1) {
        std::snprintf(name, sizeof(name), "ltx_gemm_reduce_%s_%s", msuffix(mode), es);
        c->launch(name, p.N / 64, (M + 63) / 64, 1, 256, &g, st, "splitk_reduce");
    }
}

// Dequantises the int8 projections p[i] whose buffer out[i] is set (and whose
// weights are laid out for the LDS-DMA kernels: bytes q + 128, scale words)
// into out[i], one launch per scale type; done[i] = out[i] for those, NULL
// for the rest.
static void dequant16(ltx_ctx* c, int mode, const LtxProj* const* p, void* const* out, int n, const void** done,
                      hipStream_t st) {
    for (int sf = 0; sf < 2; sf++) {  // f16 scale pairs, then f32 scales
        LtxDq16Args a{};
        int nb = 0;
        for (int i = 0; i < n; i++) {
            if (sf == 0) done[i] = nullptr;
            const LtxProj& q = *p[i];
            if (!out[i] || !q.q8 || (q.scale_f16 ? 0 : 1) != sf) continue;
            if (!q.qraw && (!q.qflip || !q.s2.p)) continue;
            const int j = a.njobs++;
            a.raw = q.qraw;  // (of one job: the isolated GEMM)
            a.q[j] = (const uint8_t*)q.q.p;
            a.s2[j] = (const uint32_t*)(q.qraw ? q.s.p : q.s2.p);
            a.out[j] = out[i];
            a.N[j] = q.N;
            a.K[j] = q.K;
            a.start[j] = nb;
            nb += (q.K / LTX_GROUP) * ((q.N + 31) / 32);
            done[i] = out[i];
        }
        if (!a.njobs) continue;
        a.start[a.njobs] = nb;
        char name[48];
        std::snprintf(name, sizeof(name), "ltx_gemm_dq16_%s%s", msuffix(mode), sf ? "_s32" : "");
        c->launch(name, nb, 1, 1, 256, &a, st, "dq16");
    }
}

static void gate16(ltx_ctx* c, int mode, const LtxProj& p, const void* A, int M, float* out, hipStream_t st) {
    LtxGateArgs g{A, mode == LTX_MODE_BF16 ? p.w_bf16.p : p.w_f16.p, (const float*)p.bias.p, out, M};
    c->launch(mode == LTX_MODE_BF16 ? "ltx_gate_bf16" : "ltx_gate_f16", (M + 15) / 16, 1, 1, 512, &g, st);
}

// Whether ltx_op_attention pads V^T (lkv no multiple of 64) for the LDS-DMA
// kernels. The padding launch costs 7 to 9 us; the any-length kernel takes about
// twice as long a round of workgroups and key tile, less where 8 divides lkv
// (it then loads V^T in 16-byte vectors) and where its last round has few
// workgroups (they have their CUs to themselves). Measured, padded against
// any-length, us, by rounds and the last one's share of the CUs (lq x lkv, f16):
// four or more: 6,145 x 16 37 : 40, 7,001 x 200 56 : 67;
// three, an eighth: 4,200 x 72 35 : 34, x 200 45 : 44, x 264 48 : 48, x 328 52 :
// 54, x 65 35 : 38; more: 5,000 x 72 37 : 37, 6,144 x 72 37 : 46, 5,000 x 50
// 33 : 33;
// two, an eighth: 2,100 x 77 26 : 22, x 130 29 : 28, x 250 32 : 34; 8 divides:
// x 72 26 : 20, x 712 54 : 54, x 968 66 : 68; up to half: 2,400 x 77 26 : 26, x
// 130 30 : 32, x 200 32 : 30, x 328 38 : 37, x 392 40 : 41; more: 4,096 x 65
// 30 : 31, x 200 38 : 35, x 264 39 : 39, x 328 42 : 43;
// one: 1,000 x 200 20 : 15, x 255 20 : 21, x 500 25 : 30.
static bool pad_pays(const ltx_ctx* c, int lq, int lkv) {
    const int nt = (lkv + 63) / 64, wgs = (lq + 255) / 256 * LTX_H;
    const int rounds = (wgs + c->num_cu - 1) / c->num_cu, last = wgs - (rounds - 1) * c->num_cu;
    const bool few = last <= c->num_cu / 8, v8 = lkv % 8 == 0;
    if (rounds >= 4) return true;
    if (rounds == 3) return nt >= (v8 && few ? 5 : 2);
    if (rounds == 2) return nt >= (v8 ? few ? 13 : last <= c->num_cu / 2 ? 6 : 5 : few ? 4 : 2);
    return nt >= (v8 ? 28 : 5);
}

// Whether the streaming attention takes 128-query workgroups: where they fit the
// chip in one round (up to 1,024 queries), so that 256-query ones would leave half
// of it idle. A workgroup of 128 takes three quarters of the other's time (the
// same K and V^T fragments for half the MFMAs). Measured, 128 against 256, us:
// 256 x 1,024 18 : 26, 512 x 512 12 : 17, 1,024 x 1,024 23 : 28, 1,024 x 128
// 8.1 : 9.7.
static bool attn_q128(const ltx_ctx* c, int lq) { return (lq + 127) / 128 * LTX_H <= c->num_cu; }

// The attention's exponent scale: softmax scale 1/sqrt(128) times log2(e).
static const float kAttnC = (float)(1.4426950408889634 / 11.313708498984761);

// oscale multiplies the normed (and roped) rows before the 16-bit rounding:
// kAttnC for Q, so the attention reads scores in exp2 units, 1 for K.
static void qknorm16(ltx_ctx* c, int mode, const void* x, int ldx, const void* w, const float* cs, const float* sn,
                     void* y, int rows, float oscale, hipStream_t st) {
    LtxQkNormArgs a{x, (const float*)w, cs, sn, y, rows, ldx, oscale, sat_of(c, mode)};
    c->launch(mode == LTX_MODE_BF16 ? "ltx_qknorm_bf16" : "ltx_qknorm_f16", rows, 1, 1, 256, &a, st);
}

// q_scaled: Q already carries kAttnC (the block path); else plain Q.
// qk_rows: Q and K as token rows [L][4096] (the block's qk-norm output);
// else head-major [32][L][128] (ltx_op_attention). vld: V^T's row stride, a
// multiple of 64 with zeros past lkv for the LDS-DMA kernels.
static void attn16(ltx_ctx* c, int mode, const void* q, const void* k, const void* vt, int vld, const float* glog,
                   void* out, int lq, int lkv, bool q_scaled, hipStream_t st, const char* label = nullptr,
                   unsigned long long* sat = nullptr, bool qk_rows = false) {
    LtxAttnArgs a{};
    a.sat = sat;
    a.q = q;
    a.k = k;
    a.q_hs = qk_rows ? LTX_HD : lq * LTX_HD;
    a.q_rs = qk_rows ? LTX_D : LTX_HD;
    a.k_hs = qk_rows ? LTX_HD : lkv * LTX_HD;
    a.k_rs = qk_rows ? LTX_D : LTX_HD;
    a.vt = vt;
    a.v_rs = vld;
    a.glog = glog;
    a.out = out;
    a.lq = lq;
    a.lkv = lkv;
    a.scale_log2 = q_scaled ? 1.0f : kAttnC;
    a.q_tiles = (lq + 255) / 256;  // 256 queries per workgroup
    char name[48];
    const int wph = std::max(1, std::min(c->num_cu / LTX_H, a.q_tiles));  // workgroups per head
    const int nt = (lkv + 63) / 64;
    const bool whole = vld == 64 * nt;  // V^T rows of whole key tiles
    if (c->attn_kv && whole && nt <= 4 && (a.q_tiles >= 2 * wph || nt < 2)) {
        // resident K/V: each workgroup loads one head's K and V^T once and
        // runs every wph-th query tile of that head (with fewer than two
        // tiles per workgroup the streaming kernel, which overlaps the K/V
        // loads with the first tiles, is faster)
        std::snprintf(name, sizeof(name), "ltx_attn_%s_kv%s", msuffix(mode), q_scaled ? "" : "_uq");
        c->launch(name, LTX_H * wph, 1, 1, 512, &a, st, label);
        return;
    }
    if (c->attn_pp && whole && nt >= 2) {
        // ping-pong kernel: at least two 64-key tiles
        const char* v = "pp";
        if (attn_q128(c, lq)) {
            a.q_tiles = (lq + 127) / 128;
            v = "pp1";
        }
        std::snprintf(name, sizeof(name), "ltx_attn_%s_%s%s", msuffix(mode), v, q_scaled ? "" : "_uq");
        c->launch(name, a.q_tiles * LTX_H, 1, 1, 512, &a, st, label);
        return;
    }
    // any key count: 8 waves of 32 queries (whole 64-key tiles: no masking)
    std::snprintf(name, sizeof(name), "ltx_attn_%s_w8%s", msuffix(mode), lkv % 64 == 0 ? "_full" : "");
    c->launch(name, a.q_tiles * LTX_H, 1, 1, 512, &a, st, label);
}

// Splits A [M][K] into the three bf16 planes at `planes`, of `bytes` (at least
// f3_planes_bytes).
static void split3(ltx_ctx* c, const float* A, int M, int K, void* planes, size_t bytes, hipStream_t st) {
    if (f3_planes_bytes(M, K) > bytes) throw Error("split3: the planes exceed their buffer");
    const size_t n = (size_t)M * K, ps = al(n * 2);
    char* p = (char*)planes;
    LtxSplit3Args a{A, (uint16_t*)p, (uint16_t*)(p + ps), (uint16_t*)(p + 2 * ps), n};
    c->launch("ltx_split3", (unsigned)((n / 8 + 255) / 256), 1, 1, 256, &a, st, "split3");
}

// f32-mode GEMM over rows [r0, r0 + N) of a (possibly fused) projection.
// planes: A's split by split3, or NULL (the f32 MFMA kernel); part: split-K
// partial sums (f3_part_bytes) or NULL.
static void gemm32(ltx_ctx* c, const LtxProj& p, int r0, int N, const float* A, int M, float* out, int epi,
                   const float* resid, LtxAda ada, int igate, int gelu, hipStream_t st, const char* label = nullptr,
                   const void* planes = nullptr, void* part = nullptr, int ksplit = 0) {
    const size_t G = p.K / LTX_GROUP;
    const void *wb, *ws = nullptr;
    if (p.q8) {
        wb = (const int8_t*)p.q.p + (size_t)r0 * p.K;
        ws = (const char*)p.s.p + (size_t)r0 * G * (p.scale_f16 ? 2 : 4);
    } else {
        wb = (const uint16_t*)p.w_bf16.p + (size_t)r0 * p.K;
    }
    const float* bias = p.bias.p ? (const float*)p.bias.p + r0 : nullptr;
    const uint32_t qxor = p.qflip ? 0u : 0x80808080u;
    auto al16 = [](const void* q) { return ((uintptr_t)q & 15) == 0; };
    if (planes && f3_shape(c, M, N, p.K) && al16(wb) && al16(out) && al16(bias) && al16(resid) && al16(ada.tstab) &&
        al16(ada.sst)) {
        LtxGemmF3Args f{};
        LtxGemmArgs& g = f.g;
        const size_t ps = al((size_t)M * p.K * 2);
        g.a = planes;
        f.a1 = (const char*)planes + ps;
        f.a2 = (const char*)planes + 2 * ps;
        g.b = wb;
        g.scales = ws;
        g.bias = bias;
        g.out = out;
        g.resid = resid;
        g.ada = ada;
        g.M = M;
        g.N = N;
        g.K = p.K;
        g.lda = p.K;
        g.ldo = N;
        g.igate = igate;
        g.gelu = gelu;
        g.out_f32 = 1;
        g.qxor = qxor;
        g.tiles_m = (M + 127) / 128;
        g.tiles_n = N / 128;
        g.ksplit = !part ? 1 : ksplit ? ksplit : gemm_ksplit(c->num_cu, M, N, p.K, 128, 128);
        g.part = (float*)part;
        const char* es = epi == LTX_EPI_RESID_GATE ? "resid" : "store";
        char name[48];
        std::snprintf(name, sizeof(name), "ltx_gemm_f3_%s_%s%s", !p.q8 ? "w16" : p.scale_f16 ? "i8f16" : "i8f32", es,
                      epi == LTX_EPI_STORE && gelu ? "_gelu" : "");
        const int nitems = g.tiles_m * g.tiles_n * g.ksplit;
        c->launch(name, std::min(nitems, c->num_cu), 1, 1, 256, &f, st, label);
        if (g.ksplit > 1) {
            std::snprintf(name, sizeof(name), "ltx_gemm_reduce_bf16_%s", es);
            c->launch(name, N / 64, (M + 63) / 64, 1, 256, &g, st, "splitk_reduce");
        }
        return;
    }
    LtxGemm32Args g{};
    g.a = A;
    g.b = wb;
    g.scales = ws;
    g.bkind = !p.q8 ? 2 : p.scale_f16 ? 1 : 0;
    g.qxor = qxor;
    g.bias = bias;
    g.out = out;
    g.resid = resid;
    g.ada = ada;
    g.M = M;
    g.N = N;
    g.K = p.K;
    g.epi = epi;
    g.gelu = gelu;
    g.igate = igate;
    if (p.K % 32) throw Error("mode F32 GEMM: K must be a multiple of 32");
    c->launch("ltx_gemm_f32", (N + 127) / 128, (M + 127) / 128, 1, 256, &g, st, label);
}

static void gate32(ltx_ctx* c, const LtxProj& p, const float* A, int M, float* out, hipStream_t st, const char* label) {
    LtxGate32Args g{A, (const uint16_t*)p.w_bf16.p, (const float*)p.bias.p, out, M};
    c->launch("ltx_gate_f32", (M + 15) / 16, 1, 1, 512, &g, st, label);
}

static void qknorm32(ltx_ctx* c, float* x, const void* w, const float* cs, const float* sn, int rows, hipStream_t st) {
    LtxQkNorm32Args a{x, (const float*)w, cs, sn, rows, LTX_D};
    c->launch("ltx_qknorm_f32", rows, 1, 1, 256, &a, st);
}

static void attn32(ltx_ctx* c, const float* q, const float* k, const float* v, const float* glog, float* out, int lq,
                   int lkv, hipStream_t st, const char* label = nullptr) {
    LtxAttn32Args a{q, k, v, glog, out, lq, lkv, 1.0f / std::sqrt(128.0f)};
    c->launch("ltx_attn_f32", (lq + 127) / 128, LTX_H, 1, 512, &a, st, label);
}

// `to` runs what it is given next only after everything enqueued so far on
// `from` (event e).
static void stream_after(hipStream_t to, hipStream_t from, hipEvent_t e) {
    HIPC(hipEventRecord(e, from));
    HIPC(hipStreamWaitEvent(to, e, 0));
}

static void set_stage(ltx_ctx* c, int id, void* p, size_t bytes) {
    c->stage_ptr[id] = p;
    c->stage_bytes[id] = bytes;
}

// Fills stage V1 (i = 0) or V2 (1) of the last forward, if it has padded rows.
void fill_stage_v(ltx_ctx* c, int i, hipStream_t st) {
    const StageV& s = c->stage_v;
    if (!s.vt[i]) return;
    LtxVtPadArgs a{(const uint16_t*)s.vt[i], (uint16_t*)s.v[i], s.n[i], vt_ld(s.n[i])};
    c->launch("ltx_vt_unpad", (s.n[i] + 511) / 512, LTX_D / 4, 1, 256, &a, st);
}

// ---- the block ------------------------------------------------------------

void block_forward(ltx_ctx* c, const ltx_block_weights* w, const float* x, const float* tstab, int K,
                   const int32_t* tidx, const float* ctxv, int S, const float* pts2, const float* cs, const float* sn,
                   int T, float* y, int mode, hipStream_t st, bool own_graph) {
    if (!w) throw Error("NULL weights");
    if (T <= 0 || S <= 0 || K <= 0) throw Error("T, S and K must be positive");
    if (!x || !tstab || !tidx || !ctxv || !pts2 || !cs || !sn || !y) throw Error("NULL tensor argument");
    if ((const void*)x == (const void*)y) throw Error("y may not alias x");
    if (mode != LTX_MODE_F16 && mode != LTX_MODE_BF16 && mode != LTX_MODE_F32) throw Error("unknown mode");
    HIPC(hipSetDevice(c->device));
    ensure_ws(c, (size_t)T, (size_t)S, mode, !is_capturing(st));
    std::memset(c->stage_ptr, 0, sizeof(c->stage_ptr));
    c->stage_v = StageV{};
    const size_t TD = (size_t)T * LTX_D, SD = (size_t)S * LTX_D;
    LtxAda ada = make_ada(w, tstab, tidx, K);
    Carve cv{(char*)c->ws.p, 0, 0, false};

    if (mode == LTX_MODE_F32) {
        Ws32 b;
        carve32(cv, b, T, S, c);
        // self-attention (ltx/block.zig:546-547, qAttn1 520-530)
        norm_mod(c, mode, x, b.n_msa, ada, T, 0, 1, st,
             mode == LTX_MODE_F16 ? (const unsigned long long*)w->f16_over.p : nullptr);
        // the GEMMs' A operands are split into bf16 planes as they are formed,
        // where the GEMM that follows (N columns) takes planes: not every
        // projection does at every token count (f3_shape)
        const void* pl = nullptr;
        auto split = [&](const void* A, int rows, int N, int K) {
            pl = b.planes && f3_shape(c, rows, N, K) ? b.planes : nullptr;
            if (pl) split3(c, (const float*)A, rows, K, b.planes, b.planes_bytes, st);
        };
        split(b.n_msa, T, LTX_D, LTX_D);
        gemm32(c, w->qkv1, 0, LTX_D, (const float*)b.n_msa, T, (float*)b.q, LTX_EPI_STORE, nullptr, ada, 0, 0, st, "gemm:qkv1", pl, b.part);
        gemm32(c, w->qkv1, LTX_D, LTX_D, (const float*)b.n_msa, T, (float*)b.k, LTX_EPI_STORE, nullptr, ada, 0, 0, st, "gemm:qkv1", pl, b.part);
        gemm32(c, w->qkv1, 2 * LTX_D, LTX_D, (const float*)b.n_msa, T, (float*)b.v, LTX_EPI_STORE, nullptr, ada, 0, 0, st, "gemm:qkv1", pl, b.part);
        gate32(c, w->g1, (const float*)b.n_msa, T, (float*)b.glog1, st, "ltx_gate:1");
        qknorm32(c, (float*)b.q, w->qn1.p, cs, sn, T, st);
        qknorm32(c, (float*)b.k, w->kn1.p, cs, sn, T, st);
        attn32(c, (const float*)b.q, (const float*)b.k, (const float*)b.v, (const float*)b.glog1, (float*)b.o1, T, T, st, "attn:self");
        split(b.o1, T, LTX_D, LTX_D);
        gemm32(c, w->o1, 0, LTX_D, (const float*)b.o1, T, (float*)b.x_sa, LTX_EPI_RESID_GATE, x, ada, 2, 0, st, "gemm:o1", pl, b.part);
        // cross-attention (ltx/block.zig:548-568)
        norm_mod(c, mode, (const float*)b.x_sa, b.attn_in, ada, T, 6, 7, st);
        LtxEncArgs ea{ctxv, (const float*)w->psst.p, pts2, b.enc, S};
        c->launch("ltx_enc_f32", S, 1, 1, 256, &ea, st);
        split(b.attn_in, T, LTX_D, LTX_D);
        gemm32(c, w->q2, 0, LTX_D, (const float*)b.attn_in, T, (float*)b.q2, LTX_EPI_STORE, nullptr, ada, 0, 0, st, "gemm:q2", pl, b.part);
        split(b.enc, S, LTX_D, LTX_D);
        gemm32(c, w->kv2, 0, LTX_D, (const float*)b.enc, S, (float*)b.k2, LTX_EPI_STORE, nullptr, ada, 0, 0, st, "gemm:kv2", pl, b.part);
        gemm32(c, w->kv2, LTX_D, LTX_D, (const float*)b.enc, S, (float*)b.v2, LTX_EPI_STORE, nullptr, ada, 0, 0, st, "gemm:kv2", pl, b.part);
        gate32(c, w->g2, (const float*)b.attn_in, T, (float*)b.glog2, st, "ltx_gate:2");
        qknorm32(c, (float*)b.q2, w->qn2.p, nullptr, nullptr, T, st);
        qknorm32(c, (float*)b.k2, w->kn2.p, nullptr, nullptr, S, st);
        attn32(c, (const float*)b.q2, (const float*)b.k2, (const float*)b.v2, (const float*)b.glog2, (float*)b.o2, T, S, st, "attn:cross");
        split(b.o2, T, LTX_D, LTX_D);
        gemm32(c, w->o2, 0, LTX_D, (const float*)b.o2, T, (float*)b.x_ca, LTX_EPI_RESID_GATE, (const float*)b.x_sa, ada, 8, 0, st, "gemm:o2", pl, b.part);
        // feed-forward (ltx/block.zig:569-573)
        norm_mod(c, mode, (const float*)b.x_ca, b.ff_in, ada, T, 3, 4, st);
        split(b.ff_in, T, LTX_FF, LTX_D);
        gemm32(c, w->f1, 0, LTX_FF, (const float*)b.ff_in, T, (float*)b.h, LTX_EPI_STORE, nullptr, ada, 0, 1, st, "gemm:ff1", pl, b.part);
        split(b.h, T, LTX_D, LTX_FF);
        gemm32(c, w->f2, 0, LTX_D, (const float*)b.h, T, y, LTX_EPI_RESID_GATE, (const float*)b.x_ca, ada, 5, 0, st, "gemm:ff2", pl, b.part);
        set_stage(c, LTX_ST_NORM_MSA, b.n_msa, TD * 4);
        set_stage(c, LTX_ST_Q1, b.q, TD * 4);
        set_stage(c, LTX_ST_K1, b.k, TD * 4);
        set_stage(c, LTX_ST_V1, b.v, TD * 4);
        set_stage(c, LTX_ST_GLOG1, b.glog1, (size_t)T * LTX_H * 4);
        set_stage(c, LTX_ST_ATTN1, b.o1, TD * 4);
        set_stage(c, LTX_ST_X_SA, b.x_sa, TD * 4);
        set_stage(c, LTX_ST_ATTN_IN, b.attn_in, TD * 4);
        set_stage(c, LTX_ST_ATTN2, b.o2, TD * 4);
        set_stage(c, LTX_ST_X_CA, b.x_ca, TD * 4);
        set_stage(c, LTX_ST_FF_IN, b.ff_in, TD * 4);
        set_stage(c, LTX_ST_FF_H, b.h, (size_t)T * LTX_FF * 4);
        set_stage(c, LTX_ST_GLOG2, b.glog2, (size_t)T * LTX_H * 4);
        set_stage(c, LTX_ST_Q2, b.q2, TD * 4);
        set_stage(c, LTX_ST_K2, b.k2, SD * 4);
        set_stage(c, LTX_ST_V2, b.v2, SD * 4);
        return;
    }

    if (mode == LTX_MODE_F16 && !(w->f16_max <= 65504.0f))
        throw Error("mode F16: weight operands beyond the f16 range (largest |q s| or |w| " +
                    std::to_string(w->f16_max) + " > 65504); run LTX_MODE_BF16");
    unsigned long long* sat = sat_of(c, mode);
    Ws16 b;
    carve16(cv, b, T, S, c, mode);
    // the int8 weights of the projections on the four-wave GEMM, dequantised
    // for this forward (qkv1, o1, q2, o2, ff1, ff2)
    const void* dq[6];
    {
        const LtxProj* ps[6] = {&w->qkv1, &w->o1, &w->q2, &w->o2, &w->f1, &w->f2};
        dequant16(c, mode, ps, b.dq, 6, dq, st);
    }
    hipStream_t sd = c->side;
    auto fail_check = [&]() {
        if (fail_in_capture()) {
            hipStreamCaptureStatus cst = hipStreamCaptureStatusNone;
            if (hipStreamIsCapturing(st, &cst) == hipSuccess && cst == hipStreamCaptureStatusActive)
                throw Error("injected failure inside a graph capture, after the second stream joined it [LTX_FAIL_CAPTURE]");
        }
    };
    // The stages of V at ragged token counts (StageV), where this forward fills
    // them, on the second stream: V1 started just behind the attention, whose
    // workgroups leave registers for it (2,970 tokens: 5 us of 1,660; ahead of the
    // q and k norms 9), or where that stream forks again anyway, behind the second
    // gate logits.
    StageV& sv = c->stage_v;
    if (b.v1 != b.vt1) sv.vt[0] = b.vt1, sv.v[0] = b.v1, sv.n[0] = T;
    if (b.v2 != b.vt2) sv.vt[1] = b.vt2, sv.v[1] = b.v2, sv.n[1] = S;
    sv.filled = c->stage_v_wanted || (!own_graph && is_capturing(st));
    // The context side of the cross-attention: K/V modulation, fused k|v
    // GEMM (split-K partial sums in `part`), on stream s.
    auto ctx_side = [&](hipStream_t s, void* part) {
        LtxEncArgs ea{ctxv, (const float*)w->psst.p, pts2, b.enc, S, sat};
        c->launch(mode == LTX_MODE_BF16 ? "ltx_enc_bf16" : "ltx_enc_f16", S, 1, 1, 256, &ea, s);
        LtxGemmArgs gk{};
        gk.out = b.k2_16;
        gk.out2 = b.vt2;
        gk.nsplit = LTX_D;
        gk.ldv = vt_ld(S);
        gk.sat = sat;
        gk.part = (float*)part;
        gemm16(c, mode, w->kv2, b.enc, S, LTX_D, LTX_EPI_QKV, gk, s, "gemm:kv2");
        if (sv.filled) fill_stage_v(c, 1, s);
    };
    // Small T (early): the side stream fills the CUs that the main chain leaves
    // idle. Where the last round of the q|k|v GEMM's tiles leaves an eighth of
    // them, it starts after the first norm: the gate logits beside that GEMM,
    // then the context side (K/V modulation, k|v GEMM with its own partial sums,
    // k norm), and later the cross-attention's gate logits beside the q2 GEMM
    // (1,024 tokens: 653 us; with the gate logits on the main stream 667, with
    // the context side from the start 669). So also beside the 16-bit-weight GEMM
    // (256 x 128 tiles), full or not: the gate logits fit its CUs (2,048 tokens,
    // unquantised: 1,030 us; 1,090 with them on the main stream). Where another
    // GEMM fills the chip, side work beside it would wait for its end and then
    // slow the q and k norms: the context side starts with the forward, beside
    // the first norm, and the gate logits run on the main stream (2,970 tokens:
    // 1,613 against 1,645 us). At 21 token counts from 300 to 4,095, f16 and bf16,
    // that line chose the faster schedule or one within 1.3 % (a last round of 224
    // tiles: the side stream faster by 1.2 to 2.3 %; of 240: no difference).
    // Large T: side work starts only after the persistent GEMMs, whose
    // one-workgroup-per-CU grids it would otherwise hold back, and ends before
    // the attentions, which it would slow as much as it gains.
    const bool early = side_early(c, (size_t)T);
    bool side_gates = !early;
    auto early_ctx = [&]() {
        ctx_side(sd, b.part2);
        qknorm16(c, mode, b.k2_16, LTX_D, w->kn2.p, nullptr, nullptr, b.kh2, S, 1.0f, sd);
    };
    if (early) {
        const int tr = tile_rows(c, T, 3 * LTX_D, LTX_D);
        const int last = (T + tr - 1) / tr * (3 * LTX_D / 256) % c->num_cu;
        const bool w16 = !w->qkv1.q8 && !x4_shape(c, mode, T, 3 * LTX_D, LTX_D, LTX_D, true);  // 256 x 128 tiles
        side_gates = w16 || (last > 0 && last <= c->num_cu - c->num_cu / 8);
        if (!side_gates) {
            stream_after(sd, st, c->side_ev[0]);
            fail_check();
            early_ctx();
        }
    }
    // self-attention: n = modulate(rms(x), ada1, ada0); fused q|k|v GEMM
    norm_mod(c, mode, x, b.n_msa, ada, T, 0, 1, st,
             mode == LTX_MODE_F16 ? (const unsigned long long*)w->f16_over.p : nullptr);
    if (early && side_gates) {
        stream_after(sd, st, c->side_ev[0]);
        fail_check();
        gate16(c, mode, w->g1, b.n_msa, T, (float*)b.glog1, sd);
        HIPC(hipEventRecord(c->side_ev[1], sd));  // glog1 ready
        early_ctx();
    } else if (early) {
        gate16(c, mode, w->g1, b.n_msa, T, (float*)b.glog1, st);
    }
    LtxGemmArgs g{};
    g.out = b.qk16;
    g.out2 = b.vt1;
    g.nsplit = 2 * LTX_D;
    g.ldv = vt_ld(T);
    g.sat = sat;
    g.part = (float*)b.part;  // split-K partial sums (small grids)
    gemm16(c, mode, w->qkv1, b.n_msa, T, LTX_D, LTX_EPI_QKV, g, st, "gemm:qkv1", dq[0]);
    if (!early) {
        // the self-attention gate logits beside the q/k norms (both read
        // only what the GEMMs above wrote)
        stream_after(sd, st, c->side_ev[0]);
        fail_check();
        gate16(c, mode, w->g1, b.n_msa, T, (float*)b.glog1, sd);
        HIPC(hipEventRecord(c->side_ev[1], sd));  // glog1 ready
    }
    {  // q and k norms + RoPE in one pass (the RoPE rows read once)
        LtxQkNorm2Args qa{b.qk16, (const float*)w->qn1.p, (const float*)w->kn1.p, cs, sn, b.qh1, b.kh1,
                          T, 2 * LTX_D, kAttnC, 1.0f, sat};
        c->launch(mode == LTX_MODE_BF16 ? "ltx_qknorm2_bf16" : "ltx_qknorm2_f16", T, 1, 1, 256, &qa, st);
    }
    if (side_gates) HIPC(hipStreamWaitEvent(st, c->side_ev[1], 0));
    const bool late_v1 = early && side_gates;
    const bool fill_v1 = sv.filled && sv.vt[0];
    if (fill_v1 && !late_v1) stream_after(sd, st, c->side_ev[4]);
    attn16(c, mode, b.qh1, b.kh1, b.vt1, vt_ld(T), (const float*)b.glog1, b.o1, T, T, true, st, "attn:self", sat, true);
    if (fill_v1 && !late_v1) fill_stage_v(c, 0, sd);
    g = LtxGemmArgs{};
    g.out = b.x_sa;
    g.resid = x;
    g.ada = ada;
    g.igate = 2;
    g.ldo = LTX_D;
    g.part = (float*)b.part;  // split-K partial sums (small grids)
    gemm16(c, mode, w->o1, b.o1, T, LTX_D, LTX_EPI_RESID_GATE, g, st, "gemm:o1", dq[1]);
    // cross-attention
    norm_mod(c, mode, (const float*)b.x_sa, b.attn_in, ada, T, 6, 7, st);
    if (early) {
        if (side_gates) stream_after(sd, st, c->side_ev[2]);
        gate16(c, mode, w->g2, b.attn_in, T, (float*)b.glog2, side_gates ? sd : st);
        if (fill_v1 && late_v1) fill_stage_v(c, 0, sd);
    }
    g = LtxGemmArgs{};
    g.out = b.q2_16;
    g.ldo = LTX_D;
    g.sat = sat;
    g.part = (float*)b.part;  // split-K partial sums (small grids)
    gemm16(c, mode, w->q2, b.attn_in, T, LTX_D, LTX_EPI_STORE, g, st, "gemm:q2", dq[2]);
    {
        // A marker after each launch from here to the cross-attention (see
        // ltx_ctx::launch): without them the gate logits below and the k|v
        // GEMM's split-K reduce beside them interleaved so badly that they
        // took 0.57 and 0.39 ms instead of 0.09 and 0.01 (28,672 tokens).
        MarkScope marks(c, T >= kMarkRows);
        if (early) {
            qknorm16(c, mode, b.q2_16, LTX_D, w->qn2.p, nullptr, nullptr, b.qh2, T, kAttnC, st);
        } else {
            // the cross-attention gate logits on the side stream, beside the
            // context side (K/V modulation, k|v GEMM) and the q and k norms
            stream_after(sd, st, c->side_ev[2]);
            gate16(c, mode, w->g2, b.attn_in, T, (float*)b.glog2, sd);
            ctx_side(st, b.part);
            qknorm16(c, mode, b.q2_16, LTX_D, w->qn2.p, nullptr, nullptr, b.qh2, T, kAttnC, st);
            qknorm16(c, mode, b.k2_16, LTX_D, w->kn2.p, nullptr, nullptr, b.kh2, S, 1.0f, st);
        }
        stream_after(st, sd, c->side_ev[3]);  // glog2, or (early) the context side, ready
        attn16(c, mode, b.qh2, b.kh2, b.vt2, vt_ld(S), (const float*)b.glog2, b.o2, T, S, true, st, "attn:cross", sat, true);
    }
    g = LtxGemmArgs{};
    g.out = b.x_ca;
    g.resid = (const float*)b.x_sa;
    g.ada = ada;
    g.igate = 8;
    g.ldo = LTX_D;
    g.part = (float*)b.part;  // split-K partial sums (small grids)
    gemm16(c, mode, w->o2, b.o2, T, LTX_D, LTX_EPI_RESID_GATE, g, st, "gemm:o2", dq[3]);
    // feed-forward
    norm_mod(c, mode, (const float*)b.x_ca, b.ff_in, ada, T, 3, 4, st);
    g = LtxGemmArgs{};
    g.out = b.h;
    g.ldo = LTX_FF;
    g.gelu = 1;
    g.sat = sat;
    g.part = (float*)b.part;  // split-K partial sums (small grids)
    gemm16(c, mode, w->f1, b.ff_in, T, LTX_D, LTX_EPI_STORE, g, st, "gemm:ff1", dq[4]);
    g = LtxGemmArgs{};
    g.out = y;
    g.resid = (const float*)b.x_ca;
    g.ada = ada;
    g.igate = 5;
    g.ldo = LTX_D;
    g.part = (float*)b.part;  // split-K partial sums (small grids)
    gemm16(c, mode, w->f2, b.h, T, LTX_FF, LTX_EPI_RESID_GATE, g, st, "gemm:ff2", dq[5]);

    set_stage(c, LTX_ST_NORM_MSA, b.n_msa, TD * 2);
    set_stage(c, LTX_ST_Q1, b.qh1, TD * 2);
    set_stage(c, LTX_ST_K1, b.kh1, TD * 2);
    set_stage(c, LTX_ST_V1, b.v1, TD * 2);
    set_stage(c, LTX_ST_GLOG1, b.glog1, (size_t)T * LTX_H * 4);
    set_stage(c, LTX_ST_ATTN1, b.o1, TD * 2);
    set_stage(c, LTX_ST_X_SA, b.x_sa, TD * 4);
    set_stage(c, LTX_ST_ATTN_IN, b.attn_in, TD * 2);
    set_stage(c, LTX_ST_ATTN2, b.o2, TD * 2);
    set_stage(c, LTX_ST_X_CA, b.x_ca, TD * 4);
    set_stage(c, LTX_ST_FF_IN, b.ff_in, TD * 2);
    set_stage(c, LTX_ST_FF_H, b.h, (size_t)T * LTX_FF * 2);
    set_stage(c, LTX_ST_GLOG2, b.glog2, (size_t)T * LTX_H * 4);
    set_stage(c, LTX_ST_Q2, b.qh2, TD * 2);
    set_stage(c, LTX_ST_K2, b.kh2, SD * 2);
    set_stage(c, LTX_ST_V2, b.v2, SD * 2);
    if (!sv.filled && !own_graph && (sv.vt[0] || sv.vt[1])) HIPC(hipEventRecord(c->stage_ev, st));
}

bool linear_q8_needs_scratch(const ltx_ctx* c, int N, int K, int mode) {
    (void)K;
    return mode != LTX_MODE_F32 && c->gemm_dma && N % 256 == 0;
}

bool linear_aligned(const void* a, const void* q, const void* bias, const void* y) {
    return (((uintptr_t)a | (uintptr_t)q | (uintptr_t)bias | (uintptr_t)y) & 15) == 0;
}

bool linear_packed(const void* a, const void* q, const void* scales, int scale_f16, const void* bias, const void* y,
                   int K) {
    return linear_aligned(a, q, bias, y) && ((uintptr_t)scales & 3) == 0 && !(scale_f16 && (K / LTX_GROUP) % 2);
}

size_t linear_part_bytes(const ltx_ctx* c, int M, int N, int K, int mode) {
    if (!linear_q8_needs_scratch(c, N, K, mode) || x4_shape(c, mode, M, N, K, K)) return 0;
    const int t = s4_shape(c, mode, M, N, K, K, true) ? 128 : 256, s = gemm_ksplit(c->num_cu, M, N, K, t, t);
    return s > 1 ? (size_t)s * M * N * 4 : 0;
}

// ltx_op_linear_q8 / _noalloc: in the 16-bit modes the kernels take the weights as
// packed (linear_packed), the four-wave kernel's dequantisation and the small-grid
// kernel up to 256 rows also the scales; else the scales are first laid out as
// words [K/128][N] in sc.pairs.
// Operands that are not linear_packed: the scale words, and the weights as bytes
// q + 128 in sc.q, which at 16,384 x 4,096 weights takes 28 us of a call (all
// written whole before the GEMM reads them).
void check_linear_q8(int M, int N, int K, int mode) {
    if (M <= 0 || N <= 0 || K <= 0 || K % 128) throw Error("bad GEMM shape (K must be a multiple of 128)");
    if (mode != LTX_MODE_F16 && mode != LTX_MODE_BF16 && mode != LTX_MODE_F32) throw Error("unknown mode");
}

void linear_q8(ltx_ctx* c, const void* a, const int8_t* q, const void* scales, int scale_f16, const float* bias,
               void* y, int out_f32, int M, int N, int K, int gelu, int mode, const LinearScratch& sc,
               hipStream_t st) {
    check_linear_q8(M, N, K, mode);
    if (!a || !q || !scales || !y) throw Error("NULL tensor argument");
    // Borrow the caller's buffers through a non-owning projection view.
    LtxProj p;
    p.N = N;
    p.K = K;
    p.q8 = true;
    p.scale_f16 = scale_f16;
    p.q.p = (void*)q;
    p.s.p = (void*)scales;
    p.bias.p = (void*)bias;
    try {
        if (mode == LTX_MODE_F32) {
            if (!out_f32) throw Error("mode F32 writes f32 output");
            LtxAda ada{};
            const bool f3 = sc.planes && linear_aligned(a, q, bias, y);
            // as many rows at a time as the scratch takes, split K as for all
            // of them (the same bits)
            const int ks = gemm_ksplit(c->num_cu, M, N, K, 128, 128), step = f3 ? sc.plane_rows : M;
            for (int r = 0; r < M; r += step) {
                const int m = std::min(step, M - r);
                const float* ar = (const float*)a + (size_t)r * K;
                if (f3) split3(c, ar, m, K, sc.planes, f3_planes_bytes(sc.plane_rows, K), st);
                gemm32(c, p, 0, N, ar, m, (float*)y + (size_t)r * N, LTX_EPI_STORE, nullptr, ada, 0, gelu, st, nullptr,
                       f3 ? sc.planes : nullptr, sc.part, ks);
            }
        } else {
            const bool scratch = linear_q8_needs_scratch(c, N, K, mode);
            const bool x4 = scratch && sc.w16 && x4_shape(c, mode, M, N, K, K);
            if (scratch) {
                p.qraw = linear_packed(a, q, scales, scale_f16, bias, y, K);
                if (!sc.pairs || (!p.qraw && !sc.q)) throw Error("linear_q8: no scratch");
                if (!p.qraw || !(x4 || (s4_shape(c, mode, M, N, K, K, true) && s4_packed_scales(M)))) {
                    // the 256 x 256 LDS-DMA kernel reads scale words [K/128][N]
                    const size_t n2 = (size_t)N * (K / LTX_GROUP);
                    LtxPairArgs pa{scales, sc.pairs, N, K / LTX_GROUP, scale_f16 ? 0 : 1};
                    c->launch("ltx_scale_pairs", (unsigned)((n2 + 255) / 256), 1, 1, 256, &pa, st);
                    p.s2.p = sc.pairs;
                }
                if (!p.qraw) {
                    // and its weights as the bytes q + 128
                    const size_t nq = (size_t)N * K / 4;
                    LtxFlipArgs fa{(const uint32_t*)q, sc.q, nq};
                    c->launch("ltx_q8_flip", (unsigned)((nq + 255) / 256), 1, 1, 256, &fa, st);
                    p.q.p = sc.q;
                    p.qflip = true;
                }
            }
            // the four-wave kernel on the weights dequantised into sc.w16
            const void* w16 = nullptr;
            if (x4) {
                const LtxProj* ps[1] = {&p};
                void* outs[1] = {sc.w16};
                dequant16(c, mode, ps, outs, 1, &w16, st);
            }
            LtxGemmArgs g{};
            g.out = y;
            g.ldo = N;
            g.gelu = gelu;
            g.out_f32 = out_f32;
            g.part = p.qraw ? (float*)sc.part : nullptr;
            gemm16(c, mode, p, a, M, K, LTX_EPI_STORE, g, st, nullptr, w16);
        }
    } catch (...) {
        p.q.p = p.s.p = p.s2.p = p.bias.p = nullptr;
        throw;
    }
    p.q.p = p.s.p = p.s2.p = p.bias.p = nullptr;
}

}  // namespace ltx


extern "C" {

int ltx_block_forward(ltx_ctx* c, const ltx_block_weights* w, const float* x, const float* tstab, int K,
                      const int32_t* tidx, const float* ctx_tokens, int S, const float* pts2, const float* cos,
                      const float* sin, int T, float* y, int mode, void* stream) {
    LTX_GUARD(c, {
        if (!c) throw ltx::Error("NULL context");
        ltx::block_forward(c, w, x, tstab, K, tidx, ctx_tokens, S, pts2, cos, sin, T, y, mode, (hipStream_t)stream);
    })
}

// A block forward captured once into a HIP graph, with its buffers bound.
struct ltx_block_graph {
    ltx_ctx* c = nullptr;
    hipGraph_t graph = nullptr;
    hipGraphExec_t exec = nullptr;
    // the captured forward's intermediates, restored for ltx_block_stage at
    // every launch
    void* stage_ptr[LTX_ST_COUNT] = {};
    uint64_t stage_bytes[LTX_ST_COUNT] = {};
    ltx::StageV stage_v;
};

int ltx_block_graph_create(ltx_ctx* c, const ltx_block_weights* w, const float* x, const float* tstab, int K,
                           const int32_t* tidx, const float* ctx_tokens, int S, const float* pts2, const float* cos,
                           const float* sin, int T, float* y, int mode, ltx_block_graph** out) {
    LTX_GUARD(c, {
        if (!c) throw ltx::Error("NULL context");
        if (!out) throw ltx::Error("NULL output handle");
        *out = nullptr;
        if (c->prof) throw ltx::Error("event profiling is on; a graph cannot capture its events");
        if (T <= 0 || S <= 0) throw ltx::Error("bad token counts");
        HIPC(hipSetDevice(c->device));
        // the workspace is sized (and allocated) before the capture, which
        // may only record launches and event waits
        ltx::ensure_ws(c, (size_t)T, (size_t)S, mode);
        hipStream_t cs = nullptr;
        HIPC(hipStreamCreateWithFlags(&cs, hipStreamNonBlocking));
        hipGraph_t graph = nullptr;
        const hipError_t eb = hipStreamBeginCapture(cs, hipStreamCaptureModeRelaxed);
        if (eb != hipSuccess) {
            (void)hipStreamDestroy(cs);
            throw ltx::Error(std::string("graph capture could not start: ") + hipGetErrorString(eb));
        }
        try {
            ltx::block_forward(c, w, x, tstab, K, tidx, ctx_tokens, S, pts2, cos, sin, T, y, mode, cs, true);
        } catch (...) {
            // A throw after the forward forked the context's second stream
            // into the capture leaves that stream capturing: join it back
            // into cs, or the capture cannot end and every later forward
            // would find the second stream still in capture mode.
            hipStreamCaptureStatus sst = hipStreamCaptureStatusNone;
            if (hipStreamIsCapturing(c->side, &sst) == hipSuccess && sst == hipStreamCaptureStatusActive &&
                hipEventRecord(c->side_ev[1], c->side) == hipSuccess)
                (void)hipStreamWaitEvent(cs, c->side_ev[1], 0);
            (void)hipStreamEndCapture(cs, &graph);
            if (graph) (void)hipGraphDestroy(graph);
            (void)hipStreamDestroy(cs);
            throw;
        }
        const hipError_t ec = hipStreamEndCapture(cs, &graph);
        (void)hipStreamDestroy(cs);
        if (ec != hipSuccess || !graph) {
            if (graph) (void)hipGraphDestroy(graph);
            throw ltx::Error(std::string("graph capture of the block forward failed: ") + hipGetErrorString(ec));
        }
        hipGraphExec_t exec = nullptr;
        const hipError_t ei = hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0);
        if (ei != hipSuccess) {
            (void)hipGraphDestroy(graph);
            throw ltx::Error(std::string("graph instantiation failed: ") + hipGetErrorString(ei));
        }
        ltx_block_graph* g = new (std::nothrow) ltx_block_graph;
        if (!g) {
            (void)hipGraphExecDestroy(exec);
            (void)hipGraphDestroy(graph);
            throw ltx::Error("out of host memory");
        }
        g->c = c;
        g->graph = graph;
        g->exec = exec;
        std::memcpy(g->stage_ptr, c->stage_ptr, sizeof(g->stage_ptr));
        std::memcpy(g->stage_bytes, c->stage_bytes, sizeof(g->stage_bytes));
        g->stage_v = c->stage_v;
        c->ws_pins++;
        *out = g;
    })
}

int ltx_block_graph_launch(ltx_block_graph* g, void* stream) {
    ltx_ctx* c = g ? g->c : nullptr;
    LTX_GUARD(c, {
        if (!g) throw ltx::Error("NULL graph");
        HIPC(hipSetDevice(c->device));
        HIPC(hipGraphLaunch(g->exec, (hipStream_t)stream));
        std::memcpy(c->stage_ptr, g->stage_ptr, sizeof(c->stage_ptr));
        std::memcpy(c->stage_bytes, g->stage_bytes, sizeof(c->stage_bytes));
        ltx::StageV& sv = c->stage_v = g->stage_v;
        if (!sv.filled && (sv.vt[0] || sv.vt[1])) {
            sv.filled = c->stage_v_wanted || ltx::is_capturing((hipStream_t)stream);
            if (!sv.filled) HIPC(hipEventRecord(c->stage_ev, (hipStream_t)stream));
            for (int i = 0; i < 2 && sv.filled; i++) ltx::fill_stage_v(c, i, (hipStream_t)stream);
        }
    })
}

void ltx_block_graph_destroy(ltx_block_graph* g) {
    if (!g) return;
    (void)hipSetDevice(g->c->device);
    if (g->exec) (void)hipGraphExecDestroy(g->exec);
    if (g->graph) (void)hipGraphDestroy(g->graph);
    g->c->ws_pins--;
    delete g;
}

// Mode F32's planes (and partial sums) take at most this of the operator
// scratch, which the context keeps: operands of more rows go in passes.
static constexpr size_t kPlanesMax = 512u << 20;

int ltx_op_linear_q8(ltx_ctx* c, const void* a, const int8_t* q, const void* scales, int scale_f16, const float* bias,
                     void* y, int out_f32, int M, int N, int K, int gelu, int mode, void* stream) {
    LTX_GUARD(c, {
        if (!c) throw ltx::Error("NULL context");
        ltx::check_linear_q8(M, N, K, mode);  // before N and K size the scratch
        HIPC(hipSetDevice(c->device));
        ltx::LinearScratch sc{};
        hipStream_t st = (hipStream_t)stream;
        // mode F32 splits A into planes (not captured: then the f32 MFMA kernel)
        ltx::ScratchUse use(c->op_scratch, st);
        if (mode == LTX_MODE_F32 && ltx::f3_shape(c, M, N, K)) {
            const int rows = ltx::f3_rows(c, M, N, K, kPlanesMax);
            const size_t part = ltx::f3_part_bytes(c, M, N, K) / M * rows, np = ltx::f3_planes_bytes(rows, K);
            if (rows && (sc.planes = use.take(np + part))) {
                sc.plane_rows = rows;
                sc.part = part ? (char*)sc.planes + np : nullptr;
            }
        }
        // 16-bit modes: split-K partial sums (not captured: then no split)
        const bool packed = ltx::linear_packed(a, q, scales, scale_f16, bias, y, K);
        if (const size_t np = packed ? ltx::linear_part_bytes(c, M, N, K, mode) : 0)
            sc.part = use.take(np);
        if (ltx::linear_q8_needs_scratch(c, N, K, mode)) {
            // scratch owned by the context, grown as needed; all that a call of
            // this shape may use, so that one call warms up for every alignment
            const size_t nq = (size_t)N * K, np = (size_t)N * (K / LTX_GROUP) * 4;
            if (c->op_q.bytes < nq) c->op_q.alloc(nq);
            if (c->op_pairs.bytes < np) c->op_pairs.alloc(np);
            sc.q = (uint32_t*)c->op_q.p;
            sc.pairs = (uint32_t*)c->op_pairs.p;
            if (ltx::x4_shape(c, mode, M, N, K, K)) {
                if (c->op_w16.bytes < 2 * nq) c->op_w16.alloc(2 * nq);
                sc.w16 = c->op_w16.p;
            }
        }
        ltx::linear_q8(c, a, q, scales, scale_f16, bias, y, out_f32, M, N, K, gelu, mode, sc, st);
    })
}

int ltx_op_attention(ltx_ctx* c, const void* q, const void* k, const void* v, const float* glog, void* out, int lq,
                     int lkv, int mode, void* stream) {
    LTX_GUARD(c, {
        if (!c) throw ltx::Error("NULL context");
        if (lq <= 0 || lkv <= 0) throw ltx::Error("bad attention lengths");
        const bool q_scaled = (mode & LTX_ATTN_Q_SCALED) != 0;
        mode &= ~LTX_ATTN_Q_SCALED;
        if (q_scaled && mode == LTX_MODE_F32) throw ltx::Error("LTX_ATTN_Q_SCALED applies to the 16-bit modes");
        HIPC(hipSetDevice(c->device));
        hipStream_t st = (hipStream_t)stream;
        if (mode == LTX_MODE_F32) {
            ltx::attn32(c, (const float*)q, (const float*)k, (const float*)v, glog, (float*)out, lq, lkv, st);
            return LTX_OK;
        }
        // V^T's rows padded to whole key tiles for the LDS-DMA kernels (not
        // captured, or with K's rows off the DMA's 16 bytes: then the any-length
        // kernel)
        const int vld = ltx::vt_ld(lkv);
        void* pad = nullptr;
        ltx::ScratchUse use(c->op_scratch, st);
        if (vld != lkv && c->attn_pp && ((uintptr_t)k & 15) == 0 && ltx::pad_pays(c, lq, lkv) &&
            (pad = use.take((size_t)LTX_D * vld * 2))) {
            LtxVtPadArgs pa{(const uint16_t*)v, (uint16_t*)pad, lkv, vld};
            c->launch("ltx_vt_pad", (vld + 511) / 512, LTX_D / 4, 1, 256, &pa, st);
        }
        ltx::attn16(c, mode, q, k, pad ? pad : v, pad ? vld : lkv, glog, out, lq, lkv, q_scaled, st);
    })
}

int ltx_op_dequant(ltx_ctx* c, const int8_t* q, const void* scales, int scale_f16, int N, int K, float* out32,
                   void* out16, int mode, void* stream) {
    LTX_GUARD(c, {
        if (!c) throw ltx::Error("NULL context");
        if (N <= 0 || K <= 0 || K % 128) throw ltx::Error("bad dequant shape");
        HIPC(hipSetDevice(c->device));
        LtxDequantArgs a{q, scales, out32, out16, N, K, scale_f16};
        size_t n = (size_t)N * K;
        c->launch(mode == LTX_MODE_BF16 ? "ltx_dequant_bf16" : "ltx_dequant_f16", (unsigned)((n / 2 + 255) / 256), 1,
                  1, 256, &a, (hipStream_t)stream);
    })
}

}  // extern "C"
